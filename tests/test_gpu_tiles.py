"""Several steps per launch on tiles (small lattices): lattices smaller than the
halo, around tile edges and around the size limits, every boundary kind and
storage, remainders and probes; equal to single steps bit for bit, in FP64 also
to the oracle."""
import numpy as np
import pytest

from lattice_boltzmann_parallel_solver_amd import Lattice
from lattice_boltzmann_parallel_solver_amd import boundary_conditions as B
from lattice_boltzmann_parallel_solver_amd import boundary_utils as G
from oracle import lbm_oracle as O

pytestmark = pytest.mark.gpu


def _boundary(kind, lx, ly, M=G, P=B):
    if kind == "couette":
        return M.couette_flow_boundary_conditions(lx, ly, 0.05, 1.1)
    if kind == "poiseuille":
        return M.poiseuille_flow_boundary_conditions(lx, ly, 0.34, 0.33)
    if kind == "poiseuille_y":
        # the fix along y (square lattices): its directions leave columns 0 and lx - 1 sideways
        m = np.zeros((lx, ly), dtype=bool)
        m[:, 0] = m[:, -1] = True
        m[0, 1] = True
        return P.periodic_with_pressure_variations(m, 0.34, 0.33)
    if kind in ("channel", "walls"):
        return M.von_karman_boundary_conditions(lx, ly, 1.0, 0.1, max(2, ly // 5), walls=kind == "walls", y_offset=1)
    return None


def _state(lx, ly):
    rng = np.random.default_rng(lx * 1000 + ly)
    rho = 1 + 0.02 * rng.random((lx, ly))
    u = 0.03 * rng.standard_normal((lx, ly, 2))
    return O.equilibrium(rho, u) * (1 + 0.01 * rng.random((lx, ly, 9))), rho, u


def _run(lx, ly, kind, storage, chunks, temporal, probe):
    lat = Lattice(lx, ly, boundary=_boundary(kind, lx, ly), storage=storage)
    if temporal is not None:
        lat.set_temporal(temporal)
    if probe:
        lat.set_probe(lx // 2, ly - 1, 14)
    lat.set_state(*_state(lx, ly))
    for n in chunks:
        lat.run(1.3, n)
    out = lat.state() + (lat.probe(14) if probe else np.zeros(1),) + (np.array(lat.moments_sum()),)
    lat.close()
    return out


SHAPES = [(1, 1, "periodic"), (1, 9, "periodic"), (9, 1, "periodic"), (2, 3, "poiseuille"), (3, 2, "couette"),
          (3, 40, "poiseuille"), (4, 5, "walls"), (6, 6, "poiseuille_y"), (5, 60, "channel"), (13, 11, "walls"),
          (20, 30, "couette"), (41, 67, "poiseuille"), (40, 40, "poiseuille_y"), (64, 32, "walls"), (97, 50, "channel"),
          (300, 7, "poiseuille"), (131, 129, "walls"), (33, 500, "couette")]


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
@pytest.mark.parametrize("lx,ly,kind", SHAPES)
def test_tiles_equal_single_steps(lx, ly, kind, storage):
    chunks = (1, 9, 8, 2, 3, 13)
    got = _run(lx, ly, kind, storage, chunks, None, True)
    want = _run(lx, ly, kind, storage, chunks, 1, True)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("lx,ly,kind", [s for s in SHAPES if s[2] != "poiseuille_y"])
def test_tiles_equal_the_oracle(lx, ly, kind):
    got = _run(lx, ly, kind, "f64", (17,), None, False)
    want = O.run(*_state(lx, ly), 1.3, 17, _boundary(kind, lx, ly, M=O))
    for a, b in zip(got, want[:3]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage,lx,ly", [("f64", 512, 512), ("f64", 513, 512), ("f32", 384, 512), ("f32", 385, 512),
                                           ("f16", 512, 384), ("f16", 769, 257), ("f64", 4, 4000), ("f32", 3000, 60)])
@pytest.mark.parametrize("kind", ["walls", "poiseuille"])
def test_size_limits(storage, lx, ly, kind):
    got = _run(lx, ly, kind, storage, (12,), None, True)
    want = _run(lx, ly, kind, storage, (12,), 1, True)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
    if kind == "walls":
        got = _run(lx, ly, kind, storage, (12,), 2, True)
        for a, b in zip(got, want):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("walls", [100, 126, 127, 140])
def test_many_classes(walls):
    """classes around the 128 that the multi-step kernels keep in LDS"""
    lx, ly = 150, 9
    rules = []
    for k in range(walls):
        m = np.zeros((lx, ly), dtype=bool)
        m[:, 0] = True
        m[k, 3] = True
        rules.append(B.moving_wall(m, np.array([0.001 * (k + 1), 0.0]), 1.0))
    out = []
    for temporal in (None, 1):
        lat = Lattice(lx, ly, boundary=G.compose(*rules), storage="f64")
        if temporal:
            lat.set_temporal(temporal)
        lat.set_state(*_state(lx, ly))
        lat.run(1.1, 11)
        out.append(lat.state())
        lat.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage,lx,ly,kind", [("f64", 1030, 1030, "poiseuille"), ("f64", 1040, 1040, "poiseuille_y"),
                                                ("f64", 2830, 1000, "poiseuille"), ("f64", 300, 4000, "poiseuille"),
                                                ("f32", 2820, 1700, "poiseuille"), ("f32", 2000, 1700, "poiseuille"),
                                                ("f32", 1800, 1800, "poiseuille_y"), ("f16", 2050, 2048, "poiseuille")])
@pytest.mark.parametrize("at", [(0, 0), (-2, -1), (2, 5)])
def test_pressure_fix_beside_sweeps(storage, lx, ly, kind, at):
    """the rows the fix reaches are put right after a sweep without it; probes in and beside them"""
    import torch

    rng = np.random.default_rng(lx + ly)
    rho = torch.from_numpy(1 + 0.02 * rng.random((lx, ly))).cuda()
    u = torch.from_numpy(0.03 * rng.standard_normal((lx, ly, 2))).cuda()
    outs = []
    for temporal in (None, 1):
        lat = Lattice(lx, ly, boundary=_boundary(kind, lx, ly), storage=storage)
        if temporal:
            lat.set_temporal(temporal)
        lat.set_probe(at[0] % lx, at[1] % ly, 20)
        lat.set_equilibrium(rho, u)
        for n in (1, 6, 5):
            lat.run(1.3, n)
        out = [torch.empty(s, dtype=torch.float64, device="cuda") for s in ((lx, ly, 9), (lx, ly), (lx, ly, 2))]
        lat.state_into(*out)
        outs.append((out, lat.probe(20)))
        lat.close()
    for a, b in zip(outs[0][0], outs[1][0]):
        assert torch.equal(a, b)
    assert np.array_equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("storage,lx,ly", [("f64", 3, 349530), ("f64", 4, 262147), ("f64", 5, 209733), ("f64", 6, 174771),
                                           ("f32", 4, 786440)])
def test_pressure_fix_of_few_long_rows(storage, lx, ly):
    """large by their columns, but too few rows for the seam's launch (it needs K + 4)"""
    test_pressure_fix_beside_sweeps(storage, lx, ly, "poiseuille", (1, 7))
