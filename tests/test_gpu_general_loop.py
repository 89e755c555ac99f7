"""Compiled code on both sides of the rule between the loop over units and
the element loop over general code, on the GPU against the oracle."""
import numpy as np
import pytest

from general_loop_cases import CELLS, cell_line
from helpers import compare_exact, random_particles
from oracle_backend import OracleBackend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('name', CELLS)
def test_lines_against_the_oracle(name):
    lg, lc = cell_line(name), cell_line(name)
    lg.build_tracker(device='cuda:0', compile=True)
    lc.build_tracker(backend=OracleBackend())
    p = random_particles(5003, seed=3, scale=1.5e-3, p0c=7e12)
    for kw in (dict(num_turns=3), dict(num_turns=2, ele_start=3, ele_stop=9),
               dict(num_turns=2, turn_by_turn_monitor=True),
               dict(num_turns=1, turn_by_turn_monitor='ONE_TURN_EBE'),
               dict(num_turns=2, backtrack=True)):
        pg, pc = p.copy(_context='cuda:0'), p.copy()
        lg.track(pg, **kw)
        lc.track(pc, **kw)
        assert not compare_exact(pg, pc), kw
        if 'turn_by_turn_monitor' in kw:
            for f in ('x', 'zeta', 'delta', 'at_turn'):
                assert np.array_equal(getattr(lg.record_last_track, f),
                                      getattr(lc.record_last_track, f), equal_nan=True), f


def test_batch_against_the_oracle():
    from xtrack_amd import BatchTracker
    names = ('off_quads', 'cavities')
    lines = [cell_line(n) for n in names]
    parts = [random_particles(300, seed=k, scale=1.5e-3, p0c=7e12) for k in range(2)]
    sets = [p.copy(_context='cuda:0') for p in parts]
    BatchTracker(lines).track(sets, num_turns=3)
    for name, p, q in zip(names, parts, sets):
        line = cell_line(name)
        line.build_tracker(backend=OracleBackend())
        w = p.copy()
        line.track(w, num_turns=3)
        assert not compare_exact(q, w)
