"""Builds libantares_amd.so for gfx950 with hipcc (cross-compiles without a GPU) and the host extension with g++.

    python -m antares_amd.build
"""
from __future__ import annotations

import glob
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
OUT = os.path.join(CSRC, 'libantares_amd.so')
CALLS_OUT = os.path.join(HERE, 'runtime', '_calls.so')

# Packed-FP32 instruction selection is switched off for all device code.  The first 14 words of a kernel's arguments are in
# registers when it starts (pointers and numbers only; a struct and what stands behind it are fetched as before), which saves the
# first trip to memory of a launch: decode step of 32 layers, four tokens 4256 -> 4141 us, int4 GEMV 4096 x 11008 6.46 -> 6.25,
# sigmoid of 4 096 000 values 6.98 -> 6.61, partition of 16 777 216 36.1 -> 35.6.  So kernels take what their first loads need first.
FLAGS = ['--offload-arch=gfx950', '-O3', '-std=c++17', '-fPIC', '-shared',
         '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', '-mllvm', '-amdgpu-kernarg-preload-count=14', '-Wno-unused-result']


def build_calls(verbose: bool = True) -> str:
    """The host-side extension (operator calls replayed in native code) against torch's C++ headers."""
    import sysconfig

    import torch
    root = os.path.dirname(torch.__file__)
    include = [os.path.join(root, 'include'), os.path.join(root, 'include', 'torch', 'csrc', 'api', 'include'), '/opt/rocm/include',
               sysconfig.get_paths()['include']]
    cmd = ['g++', '-O2', '-std=c++17', '-fPIC', '-shared', '-w', '-D__HIP_PLATFORM_AMD__', '-DUSE_ROCM',
           f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}'] + [f'-I{i}' for i in include] + \
        [os.path.join(CSRC, 'host', 'calls.cpp'), '-o', CALLS_OUT + '.tmp', f'-L{os.path.join(root, "lib")}',
         '-ltorch_python', '-ltorch_hip', '-ltorch_cpu', '-lc10_hip', '-lc10']
    if verbose:
        print('[antares_amd.build]', ' '.join(cmd), flush=True)
    p = subprocess.run(cmd, capture_output=True, text=True)
    if p.returncode != 0:
        raise RuntimeError(f'g++ failed:\n{p.stdout}\n{p.stderr}')
    os.replace(CALLS_OUT + '.tmp', CALLS_OUT)
    return CALLS_OUT


def build(verbose: bool = True) -> str:
    sources = sorted(glob.glob(os.path.join(CSRC, '*.hip')))
    cmd = ['hipcc'] + FLAGS + sources + ['-o', OUT + '.tmp', '-lhiprtc']
    if verbose:
        print('[antares_amd.build]', ' '.join(cmd), flush=True)
    p = subprocess.run(cmd, capture_output=True, text=True)
    err = '\n'.join(l for l in p.stderr.splitlines() if 'packed-fp32-ops' not in l)
    if p.returncode != 0:
        raise RuntimeError(f'hipcc failed:\n{p.stdout}\n{err}')
    if err.strip() and verbose:
        print(err)
    os.replace(OUT + '.tmp', OUT)
    build_calls(verbose)
    return OUT


if __name__ == '__main__':
    build()
    print('built', OUT)
