"""AoS record stores (equilibrium, streaming, state read-out): node counts around
a wavefront and a block, output buffers on and off a 16-byte boundary, exact
against numpy."""
import numpy as np
import pytest

from lattice_boltzmann_parallel_solver_amd import _lib
from oracle import lbm_oracle as O

pytestmark = pytest.mark.gpu


def _at_offset(torch, values, offset):
    """values in a device buffer that starts `offset` elements off its allocation, between guard values"""
    flat = torch.full((values.size + offset + 8,), -77.0, dtype=torch.float64 if values.dtype == np.float64 else torch.float32, device="cuda")
    flat[offset:offset + values.size] = torch.from_numpy(values.reshape(-1)).cuda()
    return flat


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(1, 1), (3, 21), (1, 64), (5, 13), (64, 1), (2, 129), (7, 37), (300, 3)])
def test_record_stores(shape, dtype, offset):
    import torch

    L = _lib.load()
    rng = np.random.default_rng(shape[0] * 1000 + shape[1])
    n = shape[0] * shape[1]
    code = _lib.DT_F64 if dtype == np.float64 else _lib.DT_F32
    f = rng.random(shape + (9,)).astype(dtype)
    s = torch.cuda.current_stream().cuda_stream
    src, dst = _at_offset(torch, f, offset), _at_offset(torch, np.zeros_like(f), offset)
    size = f.itemsize
    _lib.check(L.lbm_stream(src.data_ptr() + offset * size, dst.data_ptr() + offset * size, *shape, code, s))
    got = dst.cpu().numpy()
    assert np.array_equal(got[offset:offset + 9 * n].reshape(f.shape), O.streaming(f))
    assert (got[:offset] == -77).all() and (got[offset + 9 * n:] == -77).all()

    rho = 1 + 0.1 * rng.random(shape)
    u = 0.1 * rng.random(shape + (2,))
    r, v = torch.from_numpy(rho.astype(dtype)).cuda(), torch.from_numpy(u.astype(dtype)).cuda()
    dst = _at_offset(torch, np.zeros_like(f), offset)
    _lib.check(L.lbm_equilibrium(r.data_ptr(), v.data_ptr(), dst.data_ptr() + offset * size, n, code, s))
    got = dst.cpu().numpy()
    want = O.equilibrium(r.cpu().numpy().astype(np.float64), v.cpu().numpy().astype(np.float64))
    mine = got[offset:offset + 9 * n].reshape(f.shape)
    if dtype == np.float64:
        assert np.array_equal(mine, want)
    else:
        # about ten roundings of terms below 2 (weights below 1/2): 10 * 2^-24
        assert np.abs(mine - want).max() < 6e-7
    assert (got[:offset] == -77).all() and (got[offset + 9 * n:] == -77).all()
