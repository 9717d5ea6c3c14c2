#!/usr/bin/env python3
"""Builds yan_amd/csrc/libyan_gemm.so, the ahead-of-time C-ABI library (declared in include/yan_gemm.h), with
hipcc for gfx950, and yan_amd/_host_calls.<ABI of this Python>.so, the host side of repeated calls, with the host compiler against torch's
headers. Needs no GPU. `--force` rebuilds even when the libraries are newer than their sources."""
import glob
import os
import platform
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
SRC = os.path.join(HERE, 'yan_gemm_capi.hip')
OUT = os.path.join(HERE, 'libyan_gemm.so')
INCLUDE = os.path.join(ROOT, 'yan_amd', 'include')


def sources():
    return [SRC, os.path.join(ROOT, 'include', 'yan_gemm.h')] + glob.glob(os.path.join(INCLUDE, 'gemm', '*.hpp'))


def up_to_date() -> bool:
    return os.path.exists(OUT) and all(os.path.getmtime(OUT) >= os.path.getmtime(s) for s in sources())


def build(force: bool = False) -> str:
    if not force and up_to_date():
        return OUT
    hipcc = os.getenv('YAN_HIPCC_COMPILER') or os.path.join(os.getenv('ROCM_PATH', '/opt/rocm'), 'bin', 'hipcc')
    cmd = [hipcc, SRC, '-o', OUT + '.tmp', '-std=c++20', '-O3', '--offload-arch=gfx950', '-shared', '-fPIC', '-fno-gpu-rdc',
           '-fvisibility=hidden', '-Wno-unused-command-line-argument',
           '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', f'-I{INCLUDE}']
    done = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, universal_newlines=True)
    if done.returncode != 0:
        raise RuntimeError(f'hipcc failed:\n{done.stdout[-4000:]}')
    os.replace(OUT + '.tmp', OUT)
    return OUT


HOST_SRC = os.path.join(HERE, 'host_calls.cpp')
# in the file's name as Python looks for it: another Python does not load it
HOST_OUT = os.path.join(ROOT, 'yan_amd', '_host_calls' + sysconfig.get_config_var('EXT_SUFFIX'))


def built_for() -> str:
    """The torch whose object layouts are compiled in; jit_kernels/host_calls.py asks the module for it before anything else."""
    import torch
    return f'torch {torch.__version__} {torch.version.git_version}'


def host_calls_up_to_date() -> bool:
    if not os.path.exists(HOST_OUT) or os.path.getmtime(HOST_OUT) < os.path.getmtime(HOST_SRC):
        return False
    with open(HOST_OUT, 'rb') as f:
        return built_for().encode() + b'\0' in f.read()


def build_host_calls(force: bool = False) -> str:
    if platform.machine() != 'x86_64':          # it passes arguments as that ABI has it; without it every call goes through Python
        return ''
    if not force and host_calls_up_to_date():
        return HOST_OUT
    import torch
    from torch.utils import cpp_extension
    lib = os.path.join(os.path.dirname(torch.__file__), 'lib')
    cmd = [os.getenv('CXX') or 'g++', HOST_SRC, '-o', HOST_OUT + '.tmp', '-std=c++17', '-O2', '-shared', '-fPIC', f'-DYAN_BUILT_FOR="{built_for()}"',
           f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}', *(f'-isystem{p}' for p in cpp_extension.include_paths()),
           f'-I{sysconfig.get_paths()["include"]}', f'-L{lib}', '-ltorch_python', '-ltorch_cpu', '-lc10']
    done = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, universal_newlines=True)
    if done.returncode != 0:
        raise RuntimeError(f'{cmd[0]} failed:\n{done.stdout[-4000:]}')
    os.replace(HOST_OUT + '.tmp', HOST_OUT)
    return HOST_OUT


if __name__ == '__main__':
    print(build_host_calls(force='--force' in sys.argv))
    print(build(force='--force' in sys.argv))
