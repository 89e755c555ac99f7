"""Build libxtrack_amd.so in the package directory (gfx950, in-tree).

    python -m xtrack_amd.build

The kernel is compiled with -ffp-contract=off (no a*b+c fusion beyond the
explicit fma calls of the math library) and with packed FP32 disabled; the
host-side program builder is plain C++ compiled with the same contraction
setting so host-evaluated constants match device arithmetic bit for bit.
"""
import os
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG, 'csrc')
BUILD = os.path.join(PKG, '_build')
ROOT = os.path.dirname(PKG)

HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
ARCH = os.environ.get('XTM_OFFLOAD_ARCH', 'gfx950')

HIP_FLAGS = ['-O3', '-std=c++17', '-fPIC', f'--offload-arch={ARCH}', '-ffp-contract=off',
             '-fno-fast-math', '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
             '-Wno-unused-command-line-argument', f'-I{ROOT}/include', f'-I{CSRC}']
CXX_FLAGS = ['-O2', '-std=c++17', '-fPIC', '-ffp-contract=off', '-fno-fast-math',
             f'-I{ROOT}/include', f'-I{CSRC}']


def _run(cmd):
    print(' '.join(cmd), flush=True)
    subprocess.run(cmd, check=True)


# headers the generated line code includes; embedded in the library so that
# run-time compilation needs no source tree
EMBEDDED_HEADERS = (('xt_math.h', CSRC), ('xt_program.h', CSRC), ('xt_ops.h', CSRC),
                    ('xt_fast.h', CSRC),
                    ('xtrack_amd.h', os.path.join(ROOT, 'include')))
_DELIM = 'XTMHDR'


def write_embedded_headers(path):
    """C++ source defining the header names and texts for hiprtc."""
    names, texts = [], []
    for nn, dd in EMBEDDED_HEADERS:
        txt = open(os.path.join(dd, nn)).read()
        if ')' + _DELIM + '"' in txt:
            raise RuntimeError(f'{nn} contains the raw-string delimiter')
        names.append(nn)
        texts.append(txt)
    out = ['// generated by xtrack_amd/build.py: headers for run-time compilation',
           'extern const int xt_embedded_header_count;',
           'extern const char *const xt_embedded_header_names[];',
           'extern const char *const xt_embedded_header_texts[];',
           f'const int xt_embedded_header_count = {len(names)};',
           'const char *const xt_embedded_header_names[] = {' +
           ', '.join(f'"{nn}"' for nn in names) + '};',
           'const char *const xt_embedded_header_texts[] = {']
    for tt in texts:
        out.append(f'R"{_DELIM}({tt}){_DELIM}",')
    out.append('};')
    with open(path, 'w') as fh:
        fh.write('\n'.join(out) + '\n')


def build(verbose=True, out=None, extra_hip_flags=(), build_dir=None):
    BUILD_ = build_dir or BUILD
    os.makedirs(BUILD_, exist_ok=True)
    kern_o = os.path.join(BUILD_, 'xt_kernel.o')
    cxx = shutil.which('g++') or 'g++'
    emb_cpp = os.path.join(BUILD_, 'xt_embedded.cpp')
    write_embedded_headers(emb_cpp)
    # flags that change the generated code's headers travel to run-time compilation
    rtc_defs = [f for f in extra_hip_flags if f.startswith('-D')]
    _run([HIPCC, *HIP_FLAGS, *extra_hip_flags,
          '-DXTM_RTC_DEFINES="' + ' '.join(rtc_defs) + '"',
          '-c', os.path.join(CSRC, 'xt_kernel.hip'), '-o', kern_o])
    mlp_o = os.path.join(BUILD_, 'xt_mlp.o')
    _run([HIPCC, *HIP_FLAGS, *extra_hip_flags, '-c', os.path.join(CSRC, 'xt_mlp.hip'),
          '-o', mlp_o])
    objs = [kern_o, mlp_o]
    for src in ('xt_builder.cpp', 'xt_flops.cpp', 'xt_codegen.cpp', emb_cpp):
        obj = os.path.join(BUILD_, os.path.basename(src).replace('.cpp', '.o'))
        _run([cxx, *CXX_FLAGS, *rtc_defs, '-c',
              src if os.path.isabs(src) else os.path.join(CSRC, src), '-o', obj])
        objs.append(obj)
    out = out or os.path.join(PKG, 'libxtrack_amd.so')
    tmp = out + '.tmp'
    _run([HIPCC, '-shared', f'--offload-arch={ARCH}', '-fPIC', '-o', tmp, *objs,
          '-L/opt/rocm/lib', '-lhiprtc', '-Wl,-rpath,/opt/rocm/lib'])
    os.replace(tmp, out)
    return out


if __name__ == '__main__':
    build()
    sys.exit(0)
