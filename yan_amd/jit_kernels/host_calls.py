"""Repeated calls of the entry points, made in native code (`csrc/host_calls.cpp`).

The reference's entries do their checks, their plan lookup and one ctypes call in Python on every call (`yan/jit_kernels/cute_gemm.py:39-64`,
`yan/jit/runtime.py:34-68`). So does an entry here the first time it sees sizes, strides, types and devices; then it hands its launch over
(`remember_call`), and a call that agrees in all of them is made natively (`repeat_call`), from the addresses of that call. A call that does
not, or a process without the built module, takes the Python way, whose checks and errors are unchanged.

Host time of a call, Python -> native: FP8 1 x 2112 x 7168 8.5 -> 3.5 us, of which 2.5 are the launch; 16-bit 6.4 -> 3.1, from bf16 activations
14.1 -> 5.9. 256 x 832 x 455 in fp32 takes 4.7 us a call instead of 7.3, four 2 x 1984 x 4608 from bf16 activations 29 instead of 41. The first
call of each size pays 2 to 3 us for the note, which the second gets back. A call that cannot be native pays the look: 0.8 us where the scales
of a large problem are copied first, 0.2 under `YAN_SPLIT_K=0` and `YAN_TUNE_TILES=1`, whose switches are asked before anything else.
"""
import ctypes
import os

import torch

from ..jit.runtime import Runtime
from . import split_k, utils
from .heuristics import tuning_enabled

try:
    from .. import _host_calls
except ImportError:
    _host_calls = None
# (a module of another torch would read its tensors at wrong offsets; csrc/build.py compiles the name in)
if getattr(_host_calls, 'built_for', None) != f'torch {torch.__version__} {torch.version.git_version}':
    _host_calls = None

# which entry a remembered call belongs to
FP8, CAST_FP8, BF16, FP16, FLOAT, CONTIGUOUS, MASKED, PER_TOKEN, PER_BLOCK = range(1, 10)
_TENSOR, _CONSTANT, _STREAM, _WORKSPACE = range(4)
_THE_STREAM, _THE_WORKSPACE = (_STREAM, 0), (_WORKSPACE, 0)


def _never(*_) -> bool:
    return False


def setup_native() -> None:
    """Hands the native module what it looks at on every call."""
    _host_calls.setup(utils.__dict__, split_k.__dict__, os.__dict__, utils._environ, utils._environ_bytes, torch._C._cuda_getDevice,
                      torch._C._cuda_getCurrentRawStream, split_k._is_capturing)


repeat_call = _never
if _host_calls is not None and utils._environ is not None:
    try:
        setup_native()
        repeat_call = _host_calls.call
    except (AttributeError, TypeError):          # a torch without the raw accessors
        pass


def _native_parts(runtime: Runtime) -> tuple:
    """A kernel's address and what each of its arguments is (None: a float, which goes where floats go). Kept with the kernel: it is asked for
    with every size that is new."""
    kinds = tuple(_TENSOR if isinstance(kind, torch.dtype) else _STREAM if kind is torch.cuda.Stream else None if kind is float else _CONSTANT
                  for _, kind in runtime.args)
    return ctypes.cast(runtime._launch, ctypes.c_void_p).value, kinds


def remember_call(call: tuple, name: str, runtime: Runtime, args: tuple, workspace=None) -> None:
    """`call`: the entry and its arguments as `repeat_call` gets them, tensors and floats in the order of `args`, which `runtime`, the kernel
    `name`, has just been launched with. `workspace`: the split-K workspace among them, looked up anew by every call."""
    if repeat_call is _never or type(runtime) is not Runtime or runtime._launch is None or not split_k.split_k_enabled() or tuning_enabled():
        return
    if runtime.native is None:
        runtime.native = _native_parts(runtime)
    address, kinds = runtime.native
    spec, tensors = [], 0
    for arg, kind in zip(args, kinds):
        if kind is _CONSTANT:
            spec.append((_CONSTANT, arg))
        elif kind is _STREAM:
            spec.append(_THE_STREAM)
        elif kind is _TENSOR and arg is not workspace:
            spec.append((_TENSOR, tensors))
            tensors += 1
        elif kind is _TENSOR:
            spec.append(_THE_WORKSPACE)
    if tensors == sum([isinstance(a, torch.Tensor) for a in call]):
        _host_calls.remember(call, name, address, tuple(spec))
