"""Lines near the limit of functions per line code (2,048): what splitting by
unit code would push beyond it is compiled without units."""
import ctypes

import numpy as np
import pytest

import xtrack_amd as xt
from xtrack_amd import _native
from xtrack_amd.elements import build_raw_table


def _generate(els):
    """(status, source) of the line's forward code."""
    lib = _native.load()
    t, o, p = build_raw_table(els)
    h = ctypes.c_void_p()
    _native.check(lib.xtm_line_create(t.ctypes.data, o.ctypes.data, p.ctypes.data, len(t), 1.0,
                                      -1, ctypes.byref(h)))
    try:
        n = ctypes.c_int64()
        st = lib.xtm_line_generate_source_ex(h, 0, 0, None, 0, ctypes.byref(n), None)
        if st != 0:
            return st, ''
        buf = ctypes.create_string_buffer(n.value + 1)
        st = lib.xtm_line_generate_source_ex(h, 0, 0, buf, n.value + 1, ctypes.byref(n), None)
        return st, buf.value.decode()
    finally:
        lib.xtm_line_destroy(h)


def _quads(n_patterns):
    """Thick quadrupoles of both signs, each pair with its own pattern of
    error orders: one general code per pattern, two unit codes."""
    els = []
    for k in range(1, n_patterns + 1):
        knl = np.array([0.0] + [1e-3 * (1 + 1e-3 * j) * (k >> j & 1) for j in range(12)])
        for sign in (1, -1):
            els.append(xt.Quadrupole(length=0.5, k1=sign * 0.1 * (1 + 1e-5 * k), knl=knl))
    return els


@pytest.mark.parametrize('n_patterns,units', [(900, True), (1100, False), (2000, False)])
def test_compiled_with_or_without_units(n_patterns, units):
    st, src = _generate(_quads(n_patterns))
    assert st == 0
    assert ('xt::track_particle_units' in src) == units
    assert src.count('XT_GEN_FN void rec_') == (2 if units else 1) * n_patterns


def test_beyond_the_limit():
    assert _generate(_quads(2100))[0] == _native.XTM_ERR_UNSUPPORTED


def test_bends_of_many_variants_share_structures():
    """32 ring variants with as many bend strengths as cell counts: the bends
    get structure functions, however their units' guards divide them."""
    from test_batch import _free, _host_batch
    from xtrack_amd import lattices
    lines = [lattices.collider_variant(k) for k in range(32)]
    lib, handles, b = _host_batch(lines)
    try:
        n = ctypes.c_int64()
        _native.check(lib.xtm_batch_generate_source(b, 0, None, 0, ctypes.byref(n), None))
        buf = ctypes.create_string_buffer(n.value + 1)
        _native.check(lib.xtm_batch_generate_source(b, 0, buf, n.value + 1, ctypes.byref(n),
                                                    None))
    finally:
        _free(lib, handles, b)
    src = buf.value.decode()
    body = [f for f in src.split('XT_GEN_FN void rec_')[1:]]
    literal_bends = [f for f in body if 'xt::op_yoshida4(p, 0x' in f.split('\n}\n')[0]]
    assert not literal_bends
