"""Build recipe of libelara_amd.so (hipcc, gfx950 only).

Every .hip file under csrc/ is compiled on its own (in parallel) and linked into one shared library next to this
file; csrc/hostcall.cpp, the Python side's native argument checks, becomes the extension module _hostcall.  Float
flags: no FMA contraction, correctly rounded fp32 division and square root, denormals kept -- the conditions under
which the kernels are bitwise equal to the reference's CPU Adam.  Packed-fp32 instructions are disabled for device code.
"""
import os
import subprocess
import sys
import warnings
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / 'csrc'
LIB = HERE / 'libelara_amd.so'
HOST_SRC, HOST_LIB = CSRC / 'hostcall.cpp', HERE / '_hostcall.so'
HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
ARCH = 'gfx950'

CFLAGS = ['-O3', '-std=c++17', '-fPIC', f'--offload-arch={ARCH}', '-ffp-contract=off', '-fno-fast-math',
          '-fhip-fp32-correctly-rounded-divide-sqrt', '-fno-gpu-flush-denormals-to-zero',
          '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
          '-Wall', '-Wno-unused-command-line-argument', f'-I{HERE.parent / "include"}']


def sources():
    return sorted(CSRC.glob('*.hip'))


def source_hash():
    """16 hex digits identifying the library's kernel code: SHA-256 over the compile flags, the C header and every
    kernel source and device header (by name and contents).  Profile summaries record it, so that a figure measured
    on other kernels can be recognised as stale."""
    import hashlib
    h = hashlib.sha256(' '.join(CFLAGS[:-1]).encode())
    for f in [HERE.parent / 'include' / 'elara_amd.h', *sorted(CSRC.glob('*.hip')), *sorted(CSRC.glob('*.h'))]:
        h.update(f.name.encode())
        h.update(f.read_bytes())
    return h.hexdigest()[:16]


def _compile(src, obj):
    cmd = [HIPCC, *CFLAGS, '-c', str(src), '-o', str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'hipcc failed for {src.name}:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    return obj


def _build_host():
    """The extension module _hostcall (host code only) against this interpreter's torch, whose version it carries."""
    import sysconfig
    import torch
    inc, lib = Path(torch.__file__).parent / 'include', Path(torch.__file__).parent / 'lib'
    tmp = HOST_LIB.with_suffix('.so.tmp')
    cmd = [os.environ.get('CXX', 'g++'), '-O2', '-std=c++17', '-fPIC', '-shared', '-D__HIP_PLATFORM_AMD__=1',
           '-DUSE_ROCM', f'-I{inc}', f'-I{inc}/torch/csrc/api/include', '-I/opt/rocm/include',
           f'-I{sysconfig.get_paths()["include"]}', f'-DELR_TORCH_VERSION="{torch.__version__}"', str(HOST_SRC), '-o', str(tmp), f'-L{lib}', '-ltorch_python',
           '-ltorch_cpu', '-lc10', '-lc10_hip']
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'{HOST_SRC.name} failed:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    os.replace(tmp, HOST_LIB)


def build(verbose=False):
    """Compile every kernel source and link libelara_amd.so, and the host module (always rebuilds).  The library needs
    hipcc alone.  Where the host module cannot be built (no g++, no Python or torch headers) an older one is removed and
    a warning says so: the row ops' calls then take the Python checks."""
    objdir = HERE / '_build'
    objdir.mkdir(exist_ok=True)
    srcs = sources()
    objs = [objdir / (s.stem + '.o') for s in srcs]
    with ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        host = ex.submit(_build_host)
        list(ex.map(_compile, srcs, objs))
    tmp = LIB.with_suffix('.so.tmp')
    cmd = [HIPCC, '-shared', f'--offload-arch={ARCH}', '-o', str(tmp), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'link failed:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    os.replace(tmp, LIB)
    if host.exception() is not None:
        HOST_LIB.unlink(missing_ok=True)
        warnings.warn(f'{HOST_LIB.name} was not built (small row-op calls take several microseconds longer): '
                      f'{host.exception()}', stacklevel=2)
    if verbose:
        print(f'built {LIB}', file=sys.stderr)
    return LIB


if __name__ == '__main__':
    build(verbose=True)
