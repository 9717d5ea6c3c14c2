"""Loaded JIT kernels: a cache directory holding `kernel.cu`, `kernel.args`, `kernel.so`, called through ctypes.

Contract of the reference's `yan/jit/runtime.py` (`Runtime` :13-68, `RuntimeCache` :71-86): a directory is a
valid kernel iff the three files exist; the library is opened lazily on first call; every call checks the
argument count and each argument's dtype/type against `kernel.args`, then calls `launch(*cargs, &rc)` and
returns `rc`. Work is enqueued on the stream that is passed in and is not synchronised here.
"""
import ctypes
import os
from typing import Dict, Optional

import torch

from .template import ctype_map

KERNEL_FILES = ('kernel.cu', 'kernel.args', 'kernel.so')


class Runtime:
    def __init__(self, path: str) -> None:
        self.path = path
        self.lib = None
        self.args = None
        self._launch = None
        self._call = None
        self.native = None          # what the native repeat calls need of it
        assert self.is_path_valid(path), f'{path} is not a complete JIT kernel directory'

    @staticmethod
    def is_path_valid(path: str) -> bool:
        return os.path.isdir(path) and all(os.path.exists(os.path.join(path, f)) for f in KERNEL_FILES)

    def _load(self) -> None:
        self.lib = ctypes.CDLL(os.path.join(self.path, 'kernel.so'))
        self._launch = self.lib.launch
        self._launch.restype = None
        with open(os.path.join(self.path, 'kernel.args'), 'r') as f:
            # The file is a comma-joined list of ('name', type) tuples spelled with `torch` in scope.
            self.args = eval(f.read(), {'torch': torch, '__builtins__': {'bool': bool, 'int': int, 'float': float}})
        if self.args and not isinstance(self.args[0], tuple):
            self.args = (self.args,)      # a single ('name', type) pair evaluates to a flat tuple
        # Declared once so that ctypes marshals plain Python ints (device pointers, stream handles) and scalars itself.
        self._launch.argtypes = [ctype_map[dtype] for _, dtype in self.args] + [ctypes.POINTER(ctypes.c_int)]
        self._call = self._specialised_call()

    def _specialised_call(self):
        """The checks and conversions of `_checked_call` written out for this kernel's arguments, one expression each: plain
        tensors of the declared dtype, plain ints and floats, bare stream handles. Anything else (a tensor subclass, a Stream
        object, a wrong type) is left to `_checked_call`. The loop over a dozen arguments was a third of the host time of a
        decode-shape GEMM call, which is what bounds one: 1 x 2112 x 7168 in FP8, call after call, 10.0 -> 8.3 us with this and
        the cheaper look at the environment (`env_switch`), three 1 x 1216 x 1280 from bf16 activations 42.9 -> 32.5."""
        scope = {'Tensor': torch.Tensor, 'c_int': ctypes.c_int, 'launch': self._launch, 'checked_call': self._checked_call}
        names, checks, values = [], [], []
        for i, (_, dtype) in enumerate(self.args):
            a = f'a{i}'
            names.append(a)
            if isinstance(dtype, torch.dtype):
                scope[f'd{i}'] = dtype
                checks.append(f'type({a}) is Tensor and {a}.dtype is d{i}')
                values.append(f'{a}.data_ptr()')
            else:
                scope[f'd{i}'] = int if dtype is torch.cuda.Stream else dtype
                checks.append(f'type({a}) is d{i}')
                values.append(a)
        source = (f'def call({", ".join(names)}):\n'
                  f'    if {" and ".join(checks) or "True"}:\n'
                  f'        rc = c_int(0)\n'
                  f'        launch({", ".join(values + ["rc"])})\n'
                  f'        return rc.value\n'
                  f'    return checked_call({", ".join(names)})\n')
        exec(source, scope)
        return scope['call']

    def __call__(self, *args) -> int:
        if self._call is None:
            self._load()
        assert len(args) == len(self.args), f'Expected {len(self.args)} arguments, got {len(args)}'
        return self._call(*args)

    def _checked_call(self, *args) -> int:
        cargs = []
        for arg, (name, dtype) in zip(args, self.args):
            if isinstance(arg, torch.Tensor):
                assert arg.dtype == dtype, f'Expected tensor dtype `{dtype}` for `{name}`, got `{arg.dtype}`'
                cargs.append(arg.data_ptr())
            elif dtype is torch.cuda.Stream:
                # a Stream object, or its bare hipStream_t handle as an int (on ROCm `cuda_stream` is that handle)
                assert isinstance(arg, (torch.cuda.Stream, int)), f'Expected a stream for `{name}`, got `{type(arg)}`'
                cargs.append(arg if isinstance(arg, int) else arg.cuda_stream)
            else:
                assert isinstance(arg, dtype), f'Expected built-in type `{dtype}` for `{name}`, got `{type(arg)}`'
                cargs.append(arg)
        rc = ctypes.c_int(0)
        self._launch(*cargs, rc)
        return rc.value


class RuntimeCache:
    """In-process map path -> Runtime that falls back to whatever a previous process left on disk."""

    def __init__(self) -> None:
        self.cache: Dict[str, Runtime] = {}

    def __getitem__(self, path: str) -> Optional[Runtime]:
        hit = self.cache.get(path)
        if hit is None and Runtime.is_path_valid(path):
            hit = self.cache[path] = Runtime(path)
        return hit

    def __setitem__(self, path: str, runtime: Runtime) -> None:
        self.cache[path] = runtime
