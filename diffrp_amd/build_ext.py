"""
Build of the HIP library ``diffrp_amd/lib/libdrp_hip.so`` for gfx950.

hipcc compiles each ``csrc/*.hip`` file to an object and links one shared
library with a plain C ABI (``include/drp.h``).  Flags:
  -ffp-contract=off      the float operation sequence is the one written
                         (bit-exact ids / depth against a scalar CPU restatement)
  -packed-fp32-ops off   no v_pk_*_f32 instructions are generated
``diffrp_amd/lib/libdrp_autograd.so`` is host code (``csrc/drp_autograd.cpp``),
built by the host compiler against the headers of the torch it is imported with.
"""
import os
import shlex
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
OUT_DIR = os.path.join(HERE, 'lib')
LIB_PATH = os.path.join(OUT_DIR, 'libdrp_hip.so')
AUTOGRAD_LIB_PATH = os.path.join(OUT_DIR, 'libdrp_autograd.so')
ARCH = os.environ.get('DRP_OFFLOAD_ARCH', 'gfx950')

SOURCES = ['drp_raster.hip', 'drp_tribwd_attr.hip', 'drp_tribwd_fused.hip', 'drp_tribwd.hip', 'drp_interp.hip', 'drp_gather.hip',
           'drp_aa.hip', 'drp_mesh.hip', 'drp_edge.hip', 'drp_gbuffer.hip', 'drp_texture.hip', 'drp_loss.hip',
           'drp_clip.hip', 'drp_compose.hip', 'drp_fork.hip', 'drp_capi.hip']

HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
CFLAGS = [
    '-O3', '-std=c++17', '-fPIC', f'--offload-arch={ARCH}',
    '-ffp-contract=off', '-fno-fast-math',
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    '-munsafe-fp-atomics',
    '-Wall', '-Wno-unused-function', '-Wno-unused-variable',
]


def _compile(src: str) -> str:
    obj = os.path.join(OUT_DIR, os.path.splitext(src)[0] + '.o')
    cmd = [HIPCC] + CFLAGS + ['-c', os.path.join(CSRC, src), '-o', obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'hipcc failed for {src}:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    return obj


def _build_autograd() -> str:
    """``libdrp_autograd.so`` (always rebuilds)."""
    import torch
    from torch.utils import cpp_extension
    tmp = AUTOGRAD_LIB_PATH + '.tmp'
    cmd = shlex.split(os.environ.get('CXX', 'g++')) + [
        '-O2', '-std=c++17', '-fPIC', '-shared', '-Wall', f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}',
        '-I', sysconfig.get_paths()['include']]
    for p in cpp_extension.include_paths():
        cmd += ['-isystem', p]
    cmd += [os.path.join(CSRC, 'drp_autograd.cpp'), '-o', tmp]
    for p in cpp_extension.library_paths():
        cmd += ['-L', p]
    cmd += ['-ltorch_python', '-ltorch_cpu', '-lc10']
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'host build failed:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    os.replace(tmp, AUTOGRAD_LIB_PATH)
    return AUTOGRAD_LIB_PATH


def build(verbose: bool = False) -> str:
    """Compile every HIP source and link ``libdrp_hip.so``, and ``libdrp_autograd.so`` (always rebuilds)."""
    os.makedirs(OUT_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(len(SOURCES) + 1, os.cpu_count() or 1)) as ex:
        host = ex.submit(_build_autograd)
        objs = list(ex.map(_compile, SOURCES))
        host.result()
    tmp = LIB_PATH + '.tmp'
    cmd = [HIPCC, '-shared', '-fPIC', f'--offload-arch={ARCH}', '-o', tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'link failed:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    os.replace(tmp, LIB_PATH)
    for o in objs:
        os.remove(o)
    if verbose:
        print('built', LIB_PATH, AUTOGRAD_LIB_PATH)
    return LIB_PATH


if __name__ == '__main__':
    build(verbose=True)
    sys.exit(0)
