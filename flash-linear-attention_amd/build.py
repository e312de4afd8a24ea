"""Compiles csrc/*.hip into fla_hip/_C/libgdn_hip.so for gfx950 with hipcc, and csrc/host/gdn_host.cpp (host code only) into
the CPython extension fla_hip/_C/gdn_host.so with g++.

    python flash-linear-attention_amd/build.py [--force]

hipcc cross-compiles without a GPU, so this runs anywhere the ROCm toolchain is
installed.  Objects are rebuilt when their source (or a header) is newer.
"""
from __future__ import annotations

import glob
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
OUT_DIR = os.path.join(HERE, 'fla_hip', '_C')
LIB = os.path.join(OUT_DIR, 'libgdn_hip.so')
OBJ_DIR = os.path.join(HERE, 'build', 'obj')
HOST_SRC = os.path.join(CSRC, 'host', 'gdn_host.cpp')
HOST_HDR = os.path.join(CSRC, 'host', 'gdn_host_train.h')
HOST_LIB = os.path.join(OUT_DIR, 'gdn_host.so')
HOST_TORCH = os.path.join(OBJ_DIR, 'gdn_host.torch')      # the torch that HOST_LIB was built with

HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
FLAGS = [
    '--offload-arch=gfx950', '-O3', '-std=c++20', '-fPIC', '-fvisibility=default',
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    # keep MFMA accumulators in ordinary VGPRs: the state and the products are read by vector ALU
    # instructions every chunk, and the AGPR form costs a copy per register each time
    '-mllvm', '-amdgpu-mfma-vgpr-form',
    '-Wno-unused-result', '-Wno-unknown-attributes',
]


def _newer(src_list, target):
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(s) > t for s in src_list)


def _compile(src, obj):
    cmd = [HIPCC, *FLAGS, '-c', src, '-o', obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = '\n'.join(l for l in r.stderr.splitlines() if 'packed-fp32-ops' not in l)
    if r.returncode != 0:
        raise RuntimeError(f'hipcc failed for {src}:\n{err}')
    if err.strip():
        sys.stderr.write(err + '\n')


def _torch_version():
    import torch
    return torch.__version__


def _compile_host():
    import torch
    root = os.path.dirname(torch.__file__)
    cmd = ['g++', '-O2', '-std=c++17', '-fPIC', '-shared', '-fvisibility=hidden', '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1',
           f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}', f'-DGDN_TORCH_VERSION="{torch.__version__}"',
           *(f'-I{d}' for d in (f'{root}/include', f'{root}/include/torch/csrc/api/include', '/opt/rocm/include', sysconfig.get_paths()['include'])),
           HOST_SRC, '-o', HOST_LIB, f'-L{root}/lib', '-ltorch_python', '-ltorch', '-ltorch_cpu', '-lc10', '-lc10_hip', f'-Wl,-rpath,{root}/lib']
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'g++ failed for {HOST_SRC}:\n{r.stderr}')
    with open(HOST_TORCH, 'w') as f:
        f.write(torch.__version__)


def build(force: bool = False, verbose: bool = True) -> str:
    os.makedirs(OUT_DIR, exist_ok=True)
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, '*.hip')))
    hdrs = sorted(glob.glob(os.path.join(CSRC, '*.h'))) + [os.path.join(HERE, '..', 'include', 'gdn_hip.h')]
    jobs, objs = [], []
    for s in srcs:
        o = os.path.join(OBJ_DIR, os.path.basename(s)[:-4] + '.o')
        objs.append(o)
        if force or _newer([s, *hdrs], o):
            jobs.append((s, o))
    host = force or _newer([HOST_SRC, HOST_HDR, hdrs[-1]], HOST_LIB) or not os.path.exists(HOST_TORCH) or open(HOST_TORCH).read() != _torch_version()
    if verbose and (jobs or host):
        print(f'[build] compiling {len(jobs)} file(s) for gfx950' + (' and the host extension' if host else ''), flush=True)
    with ThreadPoolExecutor(max_workers=min(8, max(1, len(jobs) + host))) as ex:
        pending = [ex.submit(_compile, *a) for a in jobs]
        if host:
            pending.append(ex.submit(_compile_host))
        for p in pending:
            p.result()
    if jobs or force or _newer(objs, LIB):
        cmd = [HIPCC, '--offload-arch=gfx950', '-shared', '-fPIC', '-o', LIB, *objs]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f'link failed:\n{r.stderr}')
        if verbose:
            print(f'[build] linked {LIB}', flush=True)
    return LIB


if __name__ == '__main__':
    build(force='--force' in sys.argv)
