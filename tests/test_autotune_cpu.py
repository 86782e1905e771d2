"""autotune_lattice times its one-step candidates with one step per launch, not
with the several that a lattice without a setting may take."""
import pytest

from lattice_boltzmann_parallel_solver_amd import workloads as W


class _FakeLattice:
    def __init__(self, lx, ly, boundary=None, storage="f32", device=0):
        self.lx, self.ly, self.storage, self.device, self._program = lx, ly, storage, device, boundary
        self.temporal = 0  # no setting: the library's choice

    def set_temporal(self, steps_per_launch=2, rows_per_block=0):
        self.temporal = steps_per_launch

    def __getattr__(self, name):
        return lambda *args, **kwargs: None


@pytest.mark.parametrize("choice,two,three,want", [(0.3, 0.5, 0.4, 3), (0.3, 0.4, 0.5, 2), (0.3, 2.0, 2.0, 1)])
def test_one_step_candidates_run_single_steps(monkeypatch, choice, two, three, want):
    seconds = {0: choice, 1: 1.0, 2: two, 3: three}
    monkeypatch.setattr(W, "Lattice", _FakeLattice)
    monkeypatch.setattr(W, "_time_run", lambda lat, omega, steps: seconds[lat.temporal])
    monkeypatch.setattr(W, "_compute_units", lambda device: 256)
    monkeypatch.setattr(W, "_LATTICE_CACHE", {})
    lat = _FakeLattice(512, 64)
    assert W.autotune_lattice(lat, 1.2)[3] == want
    assert lat.temporal == want
