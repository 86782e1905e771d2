"""Every multi-step kernel against the single-step kernel, each launch's kernel
asserted on both sides.

A setting of two or more steps leaves the kernel to the library where rows are
automatic: small lattices take tiles then, and a lattice without a setting
takes whatever measured fastest.  So the side under test gets a row count or a
size that reaches its kernel, the other side one step per launch, and
`next_launch` confirms both before each run."""
import numpy as np
import pytest

from lattice_boltzmann_parallel_solver_amd import Lattice
from lattice_boltzmann_parallel_solver_amd import boundary_utils as BU
from oracle import lbm_oracle as O

pytestmark = pytest.mark.gpu


def _boundary(kind, lx, ly):
    if kind == "channel":
        return BU.von_karman_boundary_conditions(lx, ly, 1.0, 0.1, max(2, ly // 4), walls=True, y_offset=1)
    if kind == "channel_open":
        return BU.von_karman_boundary_conditions(lx, ly, 1.0, 0.1, max(2, ly // 4))
    if kind == "couette":
        return BU.couette_flow_boundary_conditions(lx, ly, 0.05, 1.0)
    if kind == "poiseuille":
        return BU.poiseuille_flow_boundary_conditions(lx, ly, 0.34, 0.33)
    return None


def _run(lx, ly, storage, kind, steps, settings, probe, capacity, kernel):
    rng = np.random.default_rng(lx * 31 + ly)
    rho = 1.0 + 0.01 * rng.standard_normal((lx, ly))
    u = 0.05 * rng.standard_normal((lx, ly, 2))
    f = O.equilibrium(rho, u) + 1e-3 * rng.standard_normal((lx, ly, 9))
    lat = Lattice(lx, ly, boundary=_boundary(kind, lx, ly), storage=storage)
    lat.set_state(f, rho, u)
    if settings is not None:
        lat.set_temporal(*settings)
    lat.set_probe(probe[0], probe[1], capacity)
    assert lat.next_launch(steps) == ("first", 1)
    lat.run(1.3, 1)
    done, reached = 1, set()
    if settings is None:
        assert lat.next_launch(14) == ("step", 1)  # too few steps to look for a tiling
    for upto in (steps // 2, steps):  # two runs, so that remainders come up
        left = upto - done
        if left > 0:
            reached.add(lat.next_launch(left)[0])
            lat.run(1.3, left)
            done = upto
    assert reached == {kernel}
    out = lat.state() + (lat.probe(),)
    lat.close()
    return out


def _equal(lx, ly, storage, kind, steps, settings, kernel, capacity=None):
    probe = (lx - 2, ly // 3)
    capacity = capacity or steps
    got = _run(lx, ly, storage, kind, steps, settings, probe, capacity, kernel)
    want = _run(lx, ly, storage, kind, steps, (1, 0), probe, capacity, "step")
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


# the row sweeps with row counts given: one row a block, a few, more than the lattice has
@pytest.mark.parametrize("rows", [1, 3, 60])
@pytest.mark.parametrize("lx,ly,storage,kind", [(24, 64, "f32", "periodic"), (3, 17, "f32", "periodic"),
                                                (33, 2048, "f32", "channel"), (31, 1024, "f64", "couette"),
                                                (9, 2100, "f64", "periodic"), (7, 4500, "f16", "periodic")])
def test_two_step_sweep(lx, ly, storage, kind, rows):
    _equal(lx, ly, storage, kind, 11, (2, rows), "sweep2")


@pytest.mark.parametrize("rows", [1, 4, 60])
@pytest.mark.parametrize("lx,ly,storage,kind,k", [(24, 64, "f32", "periodic", 3), (3, 17, "f32", "periodic", 3),
                                                  (33, 1024, "f32", "channel", 3), (4, 50, "f32", "channel", 4),
                                                  (11, 300, "f16", "channel_open", 4)])
def test_k_step_sweep(lx, ly, storage, kind, k, rows):
    _equal(lx, ly, storage, kind, 17, (k, rows), "sweepk")


# automatic rows, on lattices above the tiles' size
@pytest.mark.parametrize("lx,ly,storage,kind", [(420, 500, "f32", "channel"), (500, 420, "f16", "channel_open"),
                                                (300, 900, "f64", "couette"), (130, 1700, "f32", "channel"),
                                                (110, 2048, "f16", "couette"), (140, 2000, "f64", "channel"),
                                                (90, 2500, "f32", "channel"), (3, 90000, "f64", "periodic")])
def test_two_step_sweep_automatic_rows(lx, ly, storage, kind):
    _equal(lx, ly, storage, kind, 8, (2, 0), "sweep2")


@pytest.mark.parametrize("lx,ly,storage,kind,k", [(420, 500, "f32", "channel", 3), (200, 1024, "f32", "couette", 3),
                                                  (230, 900, "f16", "channel_open", 3), (400, 600, "f32", "channel", 4),
                                                  (500, 420, "f16", "couette", 4)])
def test_k_step_sweep_automatic_rows(lx, ly, storage, kind, k):
    _equal(lx, ly, storage, kind, 11, (k, 0), "sweepk")


@pytest.mark.parametrize("k,rows,kernel", [(2, 4, "sweep2"), (3, 4, "sweepk"), (4, 5, "sweepk"), (2, 0, "tile")])
def test_probe_ring_shorter_than_the_run(k, rows, kernel):
    _equal(30, 100, "f32", "channel", 43, (k, rows), kernel, capacity=7)


@pytest.mark.parametrize("lx,ly,storage,kind", [(20, 30, "f64", "couette"), (64, 32, "f16", "channel"),
                                                (41, 67, "f32", "poiseuille"), (3, 2, "f64", "couette")])
def test_tiles(lx, ly, storage, kind):
    _equal(lx, ly, storage, kind, 60, None, "tile")


def _kernel(lx, ly, storage, kind, temporal, steps):
    lat = Lattice(lx, ly, boundary=_boundary(kind, lx, ly), storage=storage)
    if temporal:
        lat.set_temporal(temporal)
    lat.set_equilibrium(np.ones((lx, ly)), np.zeros((lx, ly, 2)))
    lat.run(1.0, 1)
    got = lat.next_launch(steps)
    lat.close()
    return got


@pytest.mark.parametrize("storage,ly,takes", [("f32", 1536, False), ("f32", 1537, True), ("f32", 2048, True),
                                              ("f32", 2049, False), ("f64", 768, False), ("f64", 769, True),
                                              ("f64", 1024, True), ("f64", 1025, False), ("f16", 2048, False)])
def test_adjacent_columns_per_lane(storage, ly, takes):
    """seven or eight waves of adjacent columns and twelve or more rows a block"""
    assert _kernel(2830, ly, storage, "channel", 2, 9) == (("sweepv", 3) if takes else ("sweep2", 2))
    assert _kernel(2816, ly, storage, "channel", 2, 9) == ("sweep2", 2)  # eleven rows a block
    if takes:
        assert _kernel(2830, ly, storage, "couette", 2, 2) == ("sweep2", 2)


@pytest.mark.parametrize("walls,takes", [(126, True), (140, False)])
def test_adjacent_columns_and_many_classes(walls, takes):
    """up to 128 classes"""
    from lattice_boltzmann_parallel_solver_amd import boundary_conditions as B

    lx, ly = 2830, 769
    rules = []
    for k in range(walls):
        m = np.zeros((lx, ly), dtype=bool)
        m[:, 0] = True
        m[k, 3] = True
        rules.append(B.moving_wall(m, np.array([0.001 * (k + 1), 0.0]), 1.0))
    lat = Lattice(lx, ly, boundary=BU.compose(*rules))
    lat.set_equilibrium(np.ones((lx, ly)), np.zeros((lx, ly, 2)))
    lat.run(1.0, 1)
    assert lat.next_launch(9)[0] == ("sweepv" if takes else "step")
    lat.close()


def test_pressure_fix_beside_sweeps():
    assert _kernel(2048, 2048, "f64", "poiseuille", 0, 9) == ("sweep2_seam", 2)
    assert _kernel(2830, 1000, "f64", "poiseuille", 0, 9) == ("sweepv_seam", 3)
    assert _kernel(2830, 1000, "f64", "poiseuille", 0, 2) == ("step", 1)
    assert _kernel(2048, 2048, "f64", "poiseuille", 1, 9) == ("step", 1)


@pytest.mark.parametrize("shape", [(1, True, False), (2, True, False), (1, False, False), (1, True, True)])
def test_a_launch_shape_means_single_steps(shape):
    """also the default shape, called for; an explicit number of steps goes before it"""
    lat = Lattice(300, 100)
    lat.set_equilibrium(np.ones((300, 100)), np.zeros((300, 100, 2)))
    lat.run(1.0, 1)
    assert lat.next_launch(29)[0] == "tile"
    lat.set_launch(*shape)
    assert lat.next_launch(9) == ("step", 1)
    lat.set_temporal(2)
    assert lat.next_launch(29)[0] == ("tile" if shape == (1, True, False) else "sweep2")
    lat.close()


@pytest.mark.parametrize("tile", [(64, 0), (0, 1), (0, 2), (128, 1)])
@pytest.mark.parametrize("lx,ly", [(60, 100), (2830, 2048)])
def test_column_tiles_asked_for_are_kept(lx, ly, tile):
    """threads or columns per thread: both keep the two-step sweep from tiles and adjacent columns"""
    lat = Lattice(lx, ly, storage="f32")
    lat.set_equilibrium(np.ones((lx, ly)), np.zeros((lx, ly, 2)))
    lat.run(1.0, 1)
    lat.set_temporal(2)
    assert lat.next_launch(29)[0] in ("tile", "sweepv")
    lat.set_sweep_tile(*tile)
    assert lat.next_launch(29) == ("sweep2", 2)
    lat.set_sweep_tile()
    assert lat.next_launch(29)[0] in ("tile", "sweepv")
    lat.close()


def test_next_launch_refuses_what_a_run_refuses():
    from lattice_boltzmann_parallel_solver_amd._lib import LbmError

    lat = Lattice(8, 8)
    with pytest.raises(LbmError):
        lat.next_launch(1)  # no state
    lat.set_equilibrium(np.ones((8, 8)), np.zeros((8, 8, 2)))
    with pytest.raises(LbmError):
        lat.next_launch(0)
    assert lat.next_launch(1) == ("first", 1)
    lat.close()
