"""Compiled code on both sides of the rule between the loop over units and
the element loop over general code, on the host against the oracle, bit for
bit: losses inside segments, partial ranges, monitors, batches."""
import numpy as np
import pytest

import xtrack_amd as xt
from fast_path_cases import edge_particles
from general_loop_cases import CELLS, cell_line
from helpers import compare_exact, random_particles
from oracle_backend import GeneratedHostBackend, OracleBackend, generated_host_line
from test_unit_constants import host_batch_track
from xtrack_amd.elements import build_raw_table


def _both(name, p, **kw):
    out = []
    for backend in (GeneratedHostBackend(), OracleBackend()):
        line = cell_line(name)
        line.build_tracker(backend=backend)
        q = p.copy()
        line.track(q, **kw)
        out.append((line, q))
    return out


@pytest.mark.parametrize('name', CELLS)
def test_lines_against_the_oracle(name):
    line = cell_line(name)
    t, o, p = build_raw_table(line.elements)
    src = generated_host_line(t, o, p, line.get_length())[3]
    assert ('xt::track_particle_units' in src) == CELLS[name][2]
    beam = random_particles(200, seed=1, scale=1.5e-3, p0c=7e12)
    for particles in (beam, edge_particles(300, seed=2)):
        (_, a), (_, b) = _both(name, particles, num_turns=3)
        assert not compare_exact(a, b)
    lost = a.sorted_by_id()['state'] <= 0
    assert lost.any()
    for kw in (dict(num_turns=2, ele_start=3, ele_stop=9), dict(ele_start=4, num_elements=13),
               dict(num_turns=2, turn_by_turn_monitor=True),
               dict(num_turns=1, turn_by_turn_monitor='ONE_TURN_EBE')):
        (la, a), (lb, b) = _both(name, beam, **kw)
        assert not compare_exact(a, b), kw
        if 'turn_by_turn_monitor' in kw:
            for f in ('x', 'px', 'y', 'zeta', 'delta', 'at_turn', 'at_element', 'state'):
                assert np.array_equal(getattr(la.record_last_track, f),
                                      getattr(lb.record_last_track, f), equal_nan=True), (kw, f)


@pytest.mark.parametrize('names', [('off_quads', 'cavities'), ('off_quads', 'tilted_kicks')],
                         ids='-'.join)
def test_batches_against_the_oracle(names, tmp_path):
    parts = [random_particles(90, seed=k, scale=1.5e-3, p0c=7e12) for k in range(2)]
    want = []
    for name, p in zip(names, parts):
        line = cell_line(name)
        line.build_tracker(backend=OracleBackend())
        q = p.copy()
        line.track(q, num_turns=3)
        want.append(q)
    host_batch_track([lambda n=n: cell_line(n) for n in names], parts, 3, str(tmp_path))
    for a, b in zip(parts, want):
        assert not compare_exact(a, b)
