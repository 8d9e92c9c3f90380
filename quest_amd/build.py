"""Builds quest_amd/libquest_hip.so for gfx950 with hipcc (the C ABI: no torch headers, no pybind) and
quest_amd/_host.so, the CPython module over it (csrc/host.cpp: torch's C++ tensors, no device code), with the host compiler.

    python -m quest_amd.build
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
LIB_PATH = os.path.join(HERE, 'libquest_hip.so')
HOST_PATH = os.path.join(HERE, '_host.so')
SOURCES = ['rowops.hip', 'hadamard_mfma.hip', 'gemm.hip', 'gemm_big.hip', 'gemm_small.hip', 'gemm_staged.hip',
           'gemm_decode.hip', 'gemm_decode_fused.hip', 'gemm_e2m3.hip', 'gemm_e2m3_mid.hip', 'gemm_e2m3_resident.hip',
           'gemm_e2m3_split.hip', 'gemm_e2m3_fused.hip', 'dense_rows.hip', 'attention.hip', 'capi.hip']

FLAGS = [
    '--offload-arch=gfx950', '-O3', '-std=c++17', '-fPIC', '-shared',
    '-ffp-contract=off',                       # the quantiser's rounding steps must stay separate
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    '-Wall', '-Wno-unused-function',
]


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(' '.join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = '\n'.join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f'{os.path.basename(cmd[0])} failed ({res.returncode}):\n{err}')
    if verbose and err.strip():
        print(err, file=sys.stderr)


def _host_command(out: str) -> list[str]:
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get('ROCM_PATH', '/opt/rocm')
    # (the ABI of torch's own std::string, or nothing that takes one would link)
    return [os.environ.get('CXX', 'g++'), '-O2', '-std=c++17', '-fPIC', '-shared', '-Wall', '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1',
            f'-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}',
            '-isystem', os.path.join(root, 'include'), '-isystem', os.path.join(rocm, 'include'), '-isystem', sysconfig.get_paths()['include'],
            os.path.join(CSRC, 'host.cpp'), '-o', out, '-L' + os.path.join(root, 'lib'), '-lc10', '-lc10_hip', '-ltorch_cpu',
            '-ltorch_python', '-L' + HERE, '-l:libquest_hip.so', '-Wl,-rpath,$ORIGIN']


def build(verbose: bool = False, extra_flags: list[str] | None = None, jobs: int = 4) -> str:
    """Compiles every source to an object (up to `jobs` at a time), links the shared library, then the host module."""
    hipcc = os.environ.get('HIPCC', os.path.join(os.environ.get('ROCM_PATH', '/opt/rocm'), 'bin', 'hipcc'))
    flags = [f for f in FLAGS if f != '-shared'] + list(extra_flags or [])
    with tempfile.TemporaryDirectory(prefix='quest_hip_build_') as tmp:
        objs = [os.path.join(tmp, os.path.splitext(s)[0] + '.o') for s in SOURCES]
        cmds = [[hipcc, *flags, '-c', os.path.join(CSRC, s), '-o', o] for s, o in zip(SOURCES, objs)]
        with ThreadPoolExecutor(max_workers=max(1, jobs)) as pool:
            for fut in [pool.submit(_run, c, verbose) for c in cmds]:
                fut.result()
        _run([hipcc, '--offload-arch=gfx950', '-shared', '-fPIC', *objs, '-o', LIB_PATH], verbose)
    _run(_host_command(HOST_PATH), verbose)
    # (an unresolved symbol would otherwise show at the first call, as a module that seems not to be there)
    _run([sys.executable, '-c', f'import torch, importlib.util as u; s = u.spec_from_file_location("_host", {HOST_PATH!r}); s.loader.exec_module(u.module_from_spec(s))'],
         verbose)
    return LIB_PATH


if __name__ == '__main__':
    print(build(verbose=True))
