"""Every element record runs the compiled unit of its own constants, also
where records have the same general code: forward, backward and as a batch,
bit for bit against the oracle."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import xtrack_amd as xt
from helpers import compare_exact, random_particles
from oracle_backend import ROOT, GeneratedHostBackend, OracleBackend, generated_host_line
from test_backtrack_code import _both as backtrack_both, generator  # noqa: F401
from test_batch import _free, _host_batch
from unit_constant_cases import PAIRS, pair_line
from xtrack_amd import _native
from xtrack_amd.elements import build_raw_table


def _beam(n=50, seed=1):
    return random_particles(n, seed=seed, scale=1e-3, p0c=7e12)


def _oracle(make, p, **kw):
    line = make()
    line.build_tracker(backend=OracleBackend())
    q = p.copy()
    line.track(q, **kw)
    return q


@pytest.mark.parametrize('repeats', [1, 3])
@pytest.mark.parametrize('name', PAIRS)
def test_forward(name, repeats):
    line = pair_line(name, repeats)
    line.build_tracker(backend=GeneratedHostBackend())
    q = _beam()
    line.track(q, num_turns=2)
    assert not compare_exact(q, _oracle(lambda: pair_line(name, repeats), _beam(), num_turns=2))
    # more distinct records than a line of literal records only has
    t, o, p = build_raw_table(line.elements)
    _, rec, _, src, _ = generated_host_line(t, o, p, line.get_length())
    assert 'struct Key' in src


@pytest.mark.parametrize('name', PAIRS)
def test_backward(generator, name):  # noqa: F811
    (_, a), (_, b) = backtrack_both(generator, lambda: pair_line(name), _beam(), num_turns=2)
    assert not compare_exact(a, b)


def host_batch_track(make, parts, num_turns, directory):
    """The lines' generated batch code on the host: one particle set per
    line, tracked in place."""
    lines = [f() for f in make]
    lib, handles, b = _host_batch(lines)
    try:
        n = ctypes.c_int64()
        nele = np.array([len(ln.elements) for ln in lines], dtype=np.int64)
        recs = np.zeros(nele.sum(), dtype=np.int32)
        _native.check(lib.xtm_batch_generate_source(b, 0, None, 0, ctypes.byref(n),
                                                    recs.ctypes.data))
        buf = ctypes.create_string_buffer(n.value + 1)
        _native.check(lib.xtm_batch_generate_source(b, 0, buf, n.value + 1, ctypes.byref(n),
                                                    None))
        entries, progs = [], []
        for h, ne in zip(handles, nele):
            entries.append(np.zeros(ne, dtype=np.int64))
            progs.append(np.zeros(lib.xtm_line_program_size(h)))
            _native.check(lib.xtm_line_copy_entry(h, entries[-1].ctypes.data))
            _native.check(lib.xtm_line_copy_program(h, progs[-1].ctypes.data))
    finally:
        _free(lib, handles, b)
    cpp, so = os.path.join(directory, 'b.cpp'), os.path.join(directory, 'b.so')
    with open(cpp, 'w') as fh:
        fh.write(buf.value.decode())
    subprocess.run(['g++', '-O1', '-std=c++17', '-fPIC', '-shared', '-ffp-contract=off',
                    '-fno-fast-math', f'-I{ROOT}/include', f'-I{ROOT}/xtrack_amd/csrc', cpp,
                    '-o', so], check=True, capture_output=True)
    glib = ctypes.CDLL(so)
    rec_l = [np.ascontiguousarray(r) for r in np.split(recs, np.cumsum(nele)[:-1])]
    lengths = np.array([ln.get_length() for ln in lines])
    ptrs = lambda arrs: (ctypes.c_void_p * len(arrs))(*[a.ctypes.data for a in arrs])
    for k, pp in enumerate(parts):
        blocks = np.array([(0, k, pp._capacity)],
                          dtype=[('first', '<i8'), ('line', '<i4'), ('count', '<i4')])
        pst = _native.make_particles_struct(pp)
        glib.xtm_batch_host(blocks.ctypes.data_as(ctypes.c_void_p), ctypes.c_int64(1),
                            ptrs(rec_l), ptrs(entries), ptrs(progs),
                            nele.ctypes.data_as(ctypes.c_void_p),
                            lengths.ctypes.data_as(ctypes.c_void_p), ctypes.byref(pst),
                            ctypes.c_int32(num_turns), ctypes.c_uint64(0))


def test_batch(tmp_path):
    """Bends of one general code within a line and across lines."""
    make = [lambda n=n, r=r: pair_line(n, r, 0) for n in PAIRS for r in (1, 3)]
    make.append(lambda: xt.Line(elements=[
        xt.Bend(length=5.0, angle=0.007, k0=0.0, model='rot-kick-rot-high-order')] * 2))
    parts = [_beam(40, seed=k) for k in range(len(make))]
    want = [_oracle(f, pp, num_turns=2) for f, pp in zip(make, parts)]
    host_batch_track(make, parts, 2, str(tmp_path))
    for k, (pp, w) in enumerate(zip(parts, want)):
        assert not compare_exact(pp, w), k
