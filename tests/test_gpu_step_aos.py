"""lattice_boltzmann_step in one kernel: lattices around the column strips (254
columns), a row block and the smallest periodic shapes, every boundary kind,
bit for bit against the oracle."""
import numpy as np
import pytest

from lattice_boltzmann_parallel_solver_amd import boundary_utils as G
from oracle import lbm_oracle as O

pytestmark = pytest.mark.gpu


def _boundaries(kind, lx, ly):
    if kind == "periodic":
        return None, None
    if kind == "couette":
        return G.couette_flow_boundary_conditions(lx, ly, 0.05, 1.1), O.couette_flow_boundary_conditions(lx, ly, 0.05, 1.1)
    if kind == "poiseuille":
        return (G.poiseuille_flow_boundary_conditions(lx, ly, 0.34, 0.33),
                O.poiseuille_flow_boundary_conditions(lx, ly, 0.34, 0.33))
    d = max(2, ly // 5)
    return (G.von_karman_boundary_conditions(lx, ly, 1.0, 0.1, d, walls=kind == "walls", y_offset=1),
            O.von_karman_boundary_conditions(lx, ly, 1.0, 0.1, d, walls=kind == "walls", y_offset=1))


@pytest.mark.parametrize("tensors", [True, False])
@pytest.mark.parametrize("lx,ly,kind", [
    (1, 1, "periodic"), (2, 1, "periodic"), (1, 70, "periodic"), (3, 2, "couette"), (2, 5, "poiseuille"),
    (3, 64, "poiseuille"), (8, 253, "walls"), (9, 254, "channel"), (10, 255, "walls"), (5, 256, "poiseuille"),
    (6, 508, "couette"), (7, 509, "walls"), (8, 510, "poiseuille"), (1600, 30, "walls"), (801, 300, "channel")])
def test_step_matches_the_oracle(lx, ly, kind, tensors):
    import torch

    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    rng = np.random.default_rng(lx * 7 + ly)
    rho = 1 + 0.05 * rng.random((lx, ly))
    u = 0.05 * rng.standard_normal((lx, ly, 2))
    f = O.equilibrium(rho, u) * (1 + 0.01 * rng.random((lx, ly, 9)))
    mine, ref = _boundaries(kind, lx, ly)
    got = [torch.from_numpy(a).cuda() for a in (f, rho, u)] if tensors else (f, rho, u)
    want = (f, rho, u)
    for _ in range(3):
        got = lattice_boltzmann_step(*got, 1.3, mine)
        want = O.step(*want, 1.3, ref)
    if tensors:
        got = [t.cpu().numpy() for t in got]
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("walls", [62, 64, 65, 90])
def test_many_classes(walls):
    """classes around the 64 the kernel keeps in LDS (each moving wall leaves its own class on one inner node)"""
    from lattice_boltzmann_parallel_solver_amd import boundary_conditions as B
    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    lx, ly = 100, 7
    rng = np.random.default_rng(walls)
    rho = 1 + 0.05 * rng.random((lx, ly))
    u = 0.05 * rng.standard_normal((lx, ly, 2))
    f = O.equilibrium(rho, u)
    rules, refs = [], []
    for k in range(walls):
        m = np.zeros((lx, ly), dtype=bool)
        m[:, 0] = True
        m[k, 3] = True
        uw = np.array([0.001 * (k + 1), 0.0])
        rules.append(B.moving_wall(m, uw, 1.0))
        refs.append(O.moving_wall(m, uw, 1.0))

    def ref(f_pre, f_post, rho=None, u=None, f_prev=None):
        for r in refs:
            f_post = r(f_pre, f_post)
        return f_post

    got = want = (f, rho, u)
    for _ in range(2):
        got = lattice_boltzmann_step(*got, 1.1, G.compose(*rules))
        want = O.step(*want, 1.1, ref)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("lx,ly,stage_bytes", [(1, 1, 1024), (7, 5, 1024), (40, 33, 1024), (40, 33, 1 << 17), (64, 64, 49152),
                                               (101, 97, 4096)])
def test_host_arrays_through_a_small_staging_buffer(lx, ly, stage_bytes):
    """lbm_step_host with rings of a few hundred bytes to one that holds all: chunks that cut across f, rho and u"""
    import torch

    from lattice_boltzmann_parallel_solver_amd import _lib

    rng = np.random.default_rng(lx)
    rho = 1 + 0.05 * rng.random((lx, ly))
    u = 0.05 * rng.standard_normal((lx, ly, 2))
    f = O.equilibrium(rho, u) * (1 + 0.01 * rng.random((lx, ly, 9)))
    out = [np.full(a.shape, -7.0) for a in (f, rho, u)]
    work = torch.empty(24 * lx * ly, dtype=torch.float64, device="cuda")
    stage = torch.empty(stage_bytes, dtype=torch.uint8, pin_memory=True)
    _lib.check(_lib.load().lbm_step_host(None, f.ctypes.data, rho.ctypes.data, u.ctypes.data, 1.3, lx, ly,
                                         *(a.ctypes.data for a in out), work.data_ptr(), stage.data_ptr(), stage_bytes,
                                         torch.cuda.current_stream().cuda_stream))
    for a, b in zip(out, O.step(f, rho, u, 1.3, None)):
        assert np.array_equal(a, b)
