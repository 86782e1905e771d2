"""lattice_boltzmann_step on tensors: rows of few columns (blocks of consecutive
nodes) around the widths where the kernels change and the sizes of a block, and
tensors that are not plain contiguous FP64 ones on the default stream; bit for bit
against the oracle."""
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


def _inputs(lx, ly):
    rng = np.random.default_rng(lx * 7 + ly)
    rho = 1 + 0.05 * rng.random((lx, ly))
    u = 0.05 * rng.standard_normal((lx, ly, 2))
    return O.equilibrium(rho, u) * (1 + 0.01 * rng.random((lx, ly, 9))), rho, u


def _cuda(arrays):
    import torch

    return [torch.from_numpy(a).cuda() for a in arrays]


def _check(got, want):
    for a, b in zip(got, want):
        assert np.array_equal(a.cpu().numpy(), b)


# rows of one to 63 columns; fewer nodes than a block stores, one block, several
@pytest.mark.parametrize("lx,ly,kind", [
    (1, 1, "periodic"), (3, 1, "periodic"), (509, 1, "periodic"), (510, 1, "periodic"), (511, 1, "periodic"),
    (1, 2, "periodic"), (1, 30, "periodic"), (2, 2, "poiseuille"), (3, 4, "poiseuille"), (253, 2, "couette"),
    (254, 2, "poiseuille"), (1000, 3, "couette"), (701, 7, "walls"), (700, 8, "channel"), (333, 15, "poiseuille"),
    (90, 16, "walls"), (211, 17, "channel"), (5, 24, "poiseuille"), (50, 31, "walls"), (400, 32, "poiseuille"),
    (61, 33, "walls"), (100, 40, "channel"), (77, 47, "poiseuille"), (64, 48, "walls"), (33, 62, "couette"),
    (40, 63, "walls")])
def test_rows_of_few_columns(lx, ly, kind):
    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    mine, ref = _boundaries(kind, lx, ly)
    want = _inputs(lx, ly)
    got = _cuda(want)
    for _ in range(3):
        got = lattice_boltzmann_step(*got, 1.3, mine)
        want = O.step(*want, 1.3, ref)
    _check(got, want)


# the strips of wider rows: few rows, and classes around the 64 that they keep in LDS
@pytest.mark.parametrize("lx,ly,kind", [(1, 63, "periodic"), (1, 300, "periodic"), (2, 63, "poiseuille"), (2, 300, "poiseuille"),
                                        (3, 100, "couette"), (1540, 63, "walls")])
def test_strips_of_few_rows(lx, ly, kind):
    test_rows_of_few_columns(lx, ly, kind)


@pytest.mark.parametrize("walls", [62, 64, 65, 90])
def test_strips_with_many_classes(walls):
    from lattice_boltzmann_parallel_solver_amd import boundary_conditions as B
    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    lx, ly = 100, 70
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

    want = _inputs(lx, ly)
    got = _cuda(want)
    for _ in range(2):
        got = lattice_boltzmann_step(*got, 1.1, G.compose(*rules))
        want = O.step(*want, 1.1, ref)
    _check(got, want)


def _as(kind, t):
    """the values of t in a tensor that has to be copied or read with care"""
    import torch

    if kind == "offset":  # 8-byte aligned only
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
        return flat.copy_(t.reshape(-1)).view(t.shape)
    if kind == "strided":
        big = torch.empty(t.shape + (2,), dtype=t.dtype, device=t.device)
        big[..., 1] = t
        return big[..., 1]
    if kind == "transposed":
        return t.transpose(0, 1).contiguous().transpose(0, 1)
    if kind == "grad":
        return t.clone().requires_grad_()
    return t


@pytest.mark.parametrize("kind", ["offset", "strided", "transposed", "grad"])
@pytest.mark.parametrize("lx,ly", [(37, 9), (21, 300)])
def test_tensors_of_other_layouts(lx, ly, kind):
    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    mine, ref = _boundaries("walls", lx, ly)
    ins = _inputs(lx, ly)
    got = lattice_boltzmann_step(*[_as(kind, t) for t in _cuda(ins)], 1.3, mine)
    assert all(t.is_contiguous() and not t.requires_grad for t in got)
    _check(got, O.step(*ins, 1.3, ref))


@pytest.mark.parametrize("dtype", ["float32", "float16", "int64"])
def test_tensors_of_other_types_are_computed_in_fp64(dtype):
    import torch
    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    mine, ref = _boundaries("couette", 21, 40)
    f, rho, u = _cuda(_inputs(21, 40))
    if dtype == "int64":
        f = f * 40
    ins = [t.to(getattr(torch, dtype)) for t in (f, rho, u)]
    if dtype == "int64":
        ins[1] = ins[1].clamp(min=1)
    got = lattice_boltzmann_step(*ins, 1.3, mine)
    assert all(t.dtype == torch.float64 for t in got)
    _check(got, O.step(*[t.double().cpu().numpy() for t in ins], 1.3, ref))


@pytest.mark.parametrize("lx,ly", [(37, 9), (200, 300)])
def test_on_a_stream_of_the_callers(lx, ly):
    """inputs made on another stream, whose work the step follows; freed inputs and
    temporaries of it are not handed out while it runs"""
    import torch
    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    mine, ref = _boundaries("walls", lx, ly)
    want = _inputs(lx, ly)
    host = [torch.from_numpy(a).pin_memory() for a in want]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        got = [t.to("cuda", non_blocking=True) for t in host]
        for _ in range(4):
            got = [t.to(torch.float32) for t in got]  # temporaries inside the call
            got = lattice_boltzmann_step(*got, 1.2, mine)
    side.synchronize()
    for _ in range(4):
        want = O.step(*[a.astype(np.float32).astype(np.float64) for a in want], 1.2, ref)
    _check(got, want)


def test_refused_inputs():
    import torch
    from lattice_boltzmann_parallel_solver_amd.lattice_boltzmann_method import lattice_boltzmann_step

    f, rho, u = _cuda(_inputs(6, 5))
    with pytest.raises(AssertionError):
        lattice_boltzmann_step(f, rho[:5], u, 1.0)
    with pytest.raises(AssertionError):
        lattice_boltzmann_step(f[..., :8], rho, u, 1.0)
    with pytest.raises(AssertionError):
        lattice_boltzmann_step(f, rho, u[..., :1], 1.0)
    with pytest.raises(AssertionError):
        lattice_boltzmann_step(f, rho, u, 2.0)
    with pytest.raises(ValueError):
        lattice_boltzmann_step(f.cpu(), rho.cpu(), u.cpu(), 1.0)
