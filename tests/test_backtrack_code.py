"""Generated backtracking code compiled for the host against the oracle:
identical bits for every coordinate, loss record and monitor record."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import xtrack_amd as xt
from fast_path_cases import CASES, IDS, edge_particles
from helpers import compare_exact, mixed_line, random_particles, segment_line
from oracle_backend import OracleBackend
from xtrack_amd import _native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'xtrack_amd', 'csrc')


@pytest.fixture(scope='module')
def generator(tmp_path_factory):
    d = tmp_path_factory.mktemp('bt')
    so = str(d / 'gen.so')
    subprocess.run(['g++', '-O1', '-std=c++17', '-fPIC', '-shared', '-ffp-contract=off',
                    f'-I{ROOT}/include', f'-I{CSRC}',
                    os.path.join(ROOT, 'tests', 'hostcode', 'backtrack_source.cpp'),
                    f'{CSRC}/xt_builder.cpp', f'{CSRC}/xt_codegen.cpp', '-o', so], check=True)
    return ctypes.CDLL(so), d


class BacktrackHostBackend(OracleBackend):
    """Oracle forward, generated code backwards."""

    def __init__(self, generator):
        super().__init__()
        self.gen, self.dir = generator

    def prepare_line(self, types, offsets, params, line_length):
        n = len(types)
        sizes = np.zeros(2, dtype=np.int64)
        assert self.gen.xth_backtrack_source(
            ctypes.c_void_p(types.ctypes.data), ctypes.c_void_p(offsets.ctypes.data),
            ctypes.c_void_p(params.ctypes.data), ctypes.c_int64(n),
            ctypes.c_void_p(sizes.ctypes.data)) == 0
        buf = ctypes.create_string_buffer(int(sizes[0]))
        rec, entry = np.zeros(n, np.int32), np.zeros(n, np.int64)
        prog = np.zeros(sizes[1])
        self.gen.xth_backtrack_copy(buf, ctypes.c_void_p(rec.ctypes.data),
                                    ctypes.c_void_p(entry.ctypes.data),
                                    ctypes.c_void_p(prog.ctypes.data))
        cpp = self.dir / f'line{len(os.listdir(self.dir))}.cpp'
        cpp.write_text(buf.raw.decode())
        so = str(cpp)[:-4] + '.so'
        subprocess.run(['g++', '-O1', '-std=c++17', '-fPIC', '-shared', '-ffp-contract=off',
                        '-fno-fast-math', f'-I{ROOT}/include', f'-I{CSRC}', str(cpp), '-o', so],
                       check=True)
        lib = ctypes.CDLL(so)
        c = ctypes
        lib.xtm_line_host.argtypes = [c.c_void_p, c.c_void_p, c.c_void_p, c.c_double,
                                      c.POINTER(_native.XtmParticles), c.c_int32, c.c_int32,
                                      c.c_int32, c.c_int32, c.c_int32, c.c_int32,
                                      c.POINTER(_native.XtmMonitor), c.c_uint64]
        forward = super().prepare_line(types, offsets, params, line_length)
        return forward, lib, rec, entry, prog, line_length

    def track_line(self, handle, particles, num_turns, ele_start, num_ele_track, end, reset,
                   flag_monitor, monitor, flags):
        forward, lib, rec, entry, prog, length = handle
        if not int(flags) & 1:
            return super().track_line(forward, particles, num_turns, ele_start, num_ele_track,
                                      end, reset, flag_monitor, monitor, flags)
        pst = _native.make_particles_struct(particles)
        mst = _native.make_monitor_struct(monitor) if monitor is not None else None
        lib.xtm_line_host(rec.ctypes.data, entry.ctypes.data, prog.ctypes.data, length,
                          ctypes.byref(pst), int(num_turns),
                          len(rec) - int(ele_start) - int(num_ele_track), int(num_ele_track),
                          int(end), int(reset), int(flag_monitor),
                          ctypes.byref(mst) if mst is not None else None, int(flags))


def _both(generator, make, p, **kw):
    out = []
    for backend in (BacktrackHostBackend(generator), OracleBackend()):
        line = make()
        line.build_tracker(backend=backend)
        q = p.copy()
        line.track(q, backtrack=True, **kw)
        out.append((line, q))
    return out


@pytest.mark.parametrize('name,make,args', CASES, ids=IDS)
def test_edges_of_forms_and_guards(generator, name, make, args):
    for p in (edge_particles(400, seed=7), random_particles(200, seed=8, scale=8e-4, p0c=7e12)):
        (_, a), (_, b) = _both(generator, lambda: make(*args), p, num_turns=2)
        assert not compare_exact(a, b)


def test_partial_ranges_losses_and_records(generator):
    p = random_particles(300, seed=9, scale=3e-3)
    for make in (lambda: mixed_line(n_cells=2), segment_line):
        for kw in (dict(num_turns=3), dict(ele_start=5, ele_stop=25),
                   dict(num_turns=1, turn_by_turn_monitor='ONE_TURN_EBE'),
                   dict(num_turns=2, freeze_longitudinal=True)):
            (la, a), (lb, b) = _both(generator, make, p, **kw)
            assert not compare_exact(a, b), kw
            if 'turn_by_turn_monitor' in kw:
                for f in ('x', 'px', 'zeta', 'ax', 'ay', 'at_turn', 'at_element', 'state'):
                    assert np.array_equal(getattr(la.record_last_track, f),
                                          getattr(lb.record_last_track, f), equal_nan=True), f
