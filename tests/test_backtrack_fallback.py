"""A compiled line whose backtracking code cannot be loaded is tracked
backwards by the interpreter, and the call succeeds: on a stand-in for the
HIP runtime whose calls fail on request, in a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCRIPT = '''
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import xtrack_amd as xt
from xtrack_amd import _native
from xtrack_amd.elements import build_raw_table
lib = _native.load()
line = xt.Line(elements=[xt.Drift(length=1.0), xt.Multipole(knl=[0, 0.1])])
t, o, p = build_raw_table(line.elements)
h = ctypes.c_void_p()
_native.check(lib.xtm_line_create(t.ctypes.data, o.ctypes.data, p.ctypes.data, len(t), 1.0, 0,
                                  ctypes.byref(h)))
_native.check(lib.xtm_line_specialize(h, 0))
pst = _native.make_particles_struct(xt.Particles(p0c=7e12, x=[1e-3]))
def track(flags):
    _native.check(lib.xtm_track_line(h, ctypes.byref(pst), 1, 0, 2, 1, 1, 0, None,
                                     ctypes.c_uint64(flags), None))
    return stub.xth_module_kernels(), stub.xth_kernels()
got = track(0)
assert got == (1, 1), got
if sys.argv[2] != 'none':
    stub.xth_fail(sys.argv[2].encode(), 1)
got = track(1)
assert got == ((2, 2) if sys.argv[2] == 'none' else (1, 2)), got
print('ok')
'''


@pytest.fixture(scope='module')
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp('hip') / 'hip_stub.so')
    subprocess.run(['g++', '-O1', '-std=c++17', '-fPIC', '-shared', '-D__HIP_PLATFORM_AMD__',
                    '-I/opt/rocm/include',
                    os.path.join(ROOT, 'tests', 'hostcode', 'hip_stub.cpp'), '-o', so],
                   check=True)
    return so


@pytest.mark.parametrize('what', ['none', 'hipModuleLoadData', 'hipModuleGetFunction',
                                  'hipMalloc', 'hipMemcpy', 'hipStreamIsCapturing'])
def test_backtracking_without_compiled_code(stub, what):
    r = subprocess.run([sys.executable, '-c', SCRIPT, stub, what], cwd=ROOT, timeout=300,
                       capture_output=True, text=True, env=dict(os.environ, PYTHONPATH=ROOT))
    assert r.returncode == 0 and r.stdout.strip().endswith('ok'), r.stderr[-2000:]
