"""The backend call with flag_monitor = 1 and an element-by-element monitor
while tracking backwards: one record at the end of each turn, from the
interpreter and from the compiled code alike."""
import numpy as np

from helpers import compare_exact, mixed_line, random_particles
from oracle_backend import HostKernelBackend
from test_backtrack_code import BacktrackHostBackend, generator  # noqa: F401
from xtrack_amd.monitor import ParticlesMonitor


def _records(backend, ebe):
    line = mixed_line(n_cells=1, aperture=0.004)
    line.build_tracker(backend=backend)
    p = random_particles(60, seed=11, scale=2e-3)
    n = len(line.elements)
    p._arrays['at_turn'][:] = 3
    mon = ParticlesMonitor(start_at_turn=0, stop_at_turn=n + 1, num_particles=60)
    mon.ebe_mode = ebe
    backend.track_line(line.tracker._handle, p, 2, 0, n, True, True, 1, mon, 1)
    # part of a turn: no turn ends, the record is taken at the part's end
    backend.track_line(line.tracker._handle, p, 1, 3, 5, False, True, 1, mon, 1)
    return p, {f: np.array(getattr(mon, f)) for f in ('x', 'px', 'y', 'zeta', 's', 'at_turn',
                                                      'at_element', 'state', 'particle_id')}


def test_records_at_the_end_of_a_turn_back(generator):  # noqa: F811
    for ebe in (1, 0):
        p, want = _records(HostKernelBackend(), ebe)
        q, got = _records(BacktrackHostBackend(generator), ebe)
        assert not compare_exact(p, q)
        # without element-by-element mode nothing is recorded backwards
        assert (want['x'] != 0).any() == bool(ebe)
        for f in want:
            assert np.array_equal(got[f], want[f], equal_nan=True), (ebe, f)
