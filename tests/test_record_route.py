"""Element-by-element records of a compiled line are taken by the
interpreter where the line's code is the loop over units, on a stand-in for
the HIP runtime that counts launches."""
import os
import subprocess
import sys

import pytest

from test_backtrack_fallback import ROOT, stub  # noqa: F401

SCRIPT = '''
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import xtrack_amd as xt
from xtrack_amd import _native
from xtrack_amd.elements import build_raw_table
lib = _native.load()
units = sys.argv[2] == 'units'
line = xt.Line(elements=[xt.Quadrupole(length=1.0, k1=0.1 if units else 0.0)] * 2)
t, o, p = build_raw_table(line.elements)
h = ctypes.c_void_p()
_native.check(lib.xtm_line_create(t.ctypes.data, o.ctypes.data, p.ctypes.data, len(t), 2.0, 0,
                                  ctypes.byref(h)))
_native.check(lib.xtm_line_specialize(h, 0))
pst = _native.make_particles_struct(xt.Particles(p0c=7e12, x=[1e-3]))
mon = xt.ParticlesMonitor(start_at_turn=0, stop_at_turn=3, num_particles=1)
mst = _native.make_monitor_struct(mon)
out = []
for flag, back in ((0, 0), (1, 0), (2, 0), (2, 1), (0, 1)):
    before = stub.xth_module_kernels()
    mst.ebe_mode = int(flag == 2)
    _native.check(lib.xtm_track_line(h, ctypes.byref(pst), 1, 0, 2, 1, 1, flag,
                                     ctypes.byref(mst), ctypes.c_uint64(back), None))
    out.append(stub.xth_module_kernels() - before)
print(out)
'''


@pytest.mark.parametrize('kind,want', [('units', [1, 1, 0, 0, 1]), ('elements', [1, 1, 1, 0, 1])])
def test_which_kernel_records(stub, kind, want):  # noqa: F811
    r = subprocess.run([sys.executable, '-c', SCRIPT, stub, kind], cwd=ROOT, timeout=300,
                       capture_output=True, text=True, env=dict(os.environ, PYTHONPATH=ROOT))
    assert r.returncode == 0 and r.stdout.strip() == str(want), (r.stdout, r.stderr[-2000:])
