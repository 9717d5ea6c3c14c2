"""The native side of repeated calls (yan_amd/csrc/host_calls.cpp) without a GPU: the module is set up with a device, streams, workspaces and
launches of the test's own, and gets calls whose arguments are plain numbers."""
import ctypes
import os
import subprocess
import sys
import sysconfig

import pytest
import torch

from yan_amd.jit_kernels import host_calls, split_k, utils

TENSOR, CONSTANT, STREAM, WORKSPACE = range(4)
ENTRY = 1 << 20         # no entry's number


class Stage:
    """What the native module looks at, and a launch that notes what it gets."""

    def __init__(self):
        self.device, self.stream, self.capturing, self.looks = 0, 111, False, 0
        self.launched, self.code, self.failed = [], 0, []
        self.make = lambda: torch.zeros(64, dtype=torch.uint8)
        self.split_k = {'_last': (None, None), '_book': split_k.WorkspaceBook(make=self.make, clear=lambda w: None),
                        'split_k_launch_failed': self.failed.append}

        def launch(first, second, rc, *_):
            self.launched.append((first, second))
            rc[0] = self.code
        self.function = ctypes.CFUNCTYPE(None, ctypes.c_uint64, ctypes.c_uint64, ctypes.POINTER(ctypes.c_int), ctypes.c_float, ctypes.c_float)(launch)

    def look(self):
        self.looks += 1
        return self.device

    def setup(self):
        native = host_calls._host_calls
        native.setup({'_num_sms': 256}, self.split_k, os.__dict__, os.environ, os.environ._data, self.look, lambda device: self.stream,
                     lambda: self.capturing)
        native.forget()

    def remember(self, call, *spec):
        return host_calls._host_calls.remember(call, 'a_kernel', ctypes.cast(self.function, ctypes.c_void_p).value, spec)

    def call(self, *call):
        return host_calls._host_calls.call(*call)

    def take(self, stream):
        """A workspace for `stream`, as an eager launch gets it by way of Python."""
        workspace = self.split_k['_book'].get(self.device, stream)
        self.split_k['_last'] = ((self.device, stream, None), workspace)
        return workspace


@pytest.fixture
def stage(monkeypatch):
    assert host_calls._host_calls is not None, 'yan_amd/csrc/build.py builds it'
    for name in ('YAN_SPLIT_K', 'YAN_TUNE_TILES'):
        monkeypatch.delenv(name, raising=False)
    stage = Stage()
    stage.setup()
    yield stage
    host_calls.setup_native()
    host_calls._host_calls.forget()


@pytest.mark.parametrize('workspace', [False, True])
def test_a_launch_that_reports_an_error_is_not_made_twice(stage, workspace):
    """The code may be an older error's, behind a launch that ran: the call raises what the Python way raises, and the workspace is marked."""
    held = stage.take(111)
    token = stage.split_k['_last'][0]
    assert stage.remember((ENTRY, 1.0), (WORKSPACE if workspace else CONSTANT, 5), (STREAM, 0))
    assert stage.call(ENTRY, 1.0) is True and stage.launched == [(held.data_ptr() if workspace else 5, 111)]
    stage.code = 98
    with pytest.raises(AssertionError, match='a_kernel failed with HIP error 98'):
        stage.call(ENTRY, 1.0)
    assert len(stage.launched) == 2 and stage.failed == ([token] if workspace else [])
    stage.code = 0
    assert stage.call(ENTRY, 1.0) is True and len(stage.launched) == 3


@pytest.mark.parametrize('when', ['stream', 'capturing'])
def test_a_launch_outlives_what_runs_while_it_is_prepared(stage, when):
    """Python code that runs between the look into the table and the launch (a finaliser, another thread) may clear and refill the table."""
    held = stage.take(111)
    assert stage.remember((ENTRY, 1.0), (CONSTANT, 5), (WORKSPACE, 0))

    def meddle(answer):
        host_calls._host_calls.forget()
        for i in range(64):
            assert stage.remember((ENTRY, i), (CONSTANT, 1000 + i), (CONSTANT, 7))
        return answer

    look = {'stream': lambda device: 111, 'capturing': lambda: False}
    look[when] = lambda *_, plain=look[when]: meddle(plain(*_))
    host_calls._host_calls.setup({'_num_sms': 256}, stage.split_k, os.__dict__, os.environ, os.environ._data, stage.look, look['stream'],
                                 look['capturing'])
    assert stage.call(ENTRY, 1.0) is True and stage.launched == [(5, held.data_ptr())]


def test_streams_in_turn_are_served_from_their_workspaces(stage):
    """Each stream gets the workspace the book holds for it, whichever stream was served last; a stream without one, one whose last launch
    failed and a capture go back to Python."""
    first, second = stage.take(111), stage.take(222)
    assert stage.remember((ENTRY, 1.0), (WORKSPACE, 0), (STREAM, 0))
    for stream in (111, 222, 111, 111, 222):
        stage.stream = stream
        assert stage.call(ENTRY, 1.0) is True
        assert stage.launched[-1] == ((first if stream == 111 else second).data_ptr(), stream)
    stage.stream = 333
    assert stage.call(ENTRY, 1.0) is False
    stage.device, stage.stream = 1, 111
    assert stage.call(ENTRY, 1.0) is False
    stage.device, stage.capturing = 0, True
    assert stage.call(ENTRY, 1.0) is False
    stage.capturing, stage.code = False, 98
    with pytest.raises(AssertionError):
        stage.call(ENTRY, 1.0)
    assert stage.failed == [(0, 111, None)]
    stage.split_k['_book'].launch_failed(*stage.failed[0])
    assert stage.call(ENTRY, 1.0) is False and len(stage.launched) == 6
    stage.stream, stage.code = 222, 0
    assert stage.call(ENTRY, 1.0) is True


@pytest.mark.parametrize('name,value', [('YAN_SPLIT_K', '0'), ('YAN_TUNE_TILES', '1')])
def test_calls_under_a_switch_cost_no_description(stage, name, value, monkeypatch):
    assert stage.remember((ENTRY, 1.0), (CONSTANT, 5), (STREAM, 0))
    looks = stage.looks
    monkeypatch.setenv(name, value)
    assert stage.call(ENTRY, 1.0) is False and stage.looks == looks
    monkeypatch.delenv(name)
    assert stage.call(ENTRY, 1.0) is True and stage.looks > looks


def test_a_module_of_another_torch_is_not_used(repo_root):
    """Neither loaded over nor kept by the build: the name of the torch is compiled in, that of the Python is in the file's name."""
    code = """
import torch
torch.__version__ = {version}
import yan_amd
from yan_amd.jit_kernels import host_calls
import importlib.util
spec = importlib.util.spec_from_file_location('build', 'yan_amd/csrc/build.py')
build = importlib.util.module_from_spec(spec)
spec.loader.exec_module(build)
print(host_calls._host_calls is not None, host_calls.repeat_call is not host_calls._never, build.host_calls_up_to_date())
"""
    for version, used in (('torch.__version__', True), ('"2.0.1+other"', False)):
        done = subprocess.run([sys.executable, '-c', code.format(version=version)], stdout=subprocess.PIPE, universal_newlines=True, check=True,
                              cwd=repo_root)
        assert done.stdout.split() == [str(used)] * 3
    assert host_calls._host_calls.__file__.endswith('_host_calls' + sysconfig.get_config_var('EXT_SUFFIX'))


@pytest.mark.parametrize('entry', ['plain', 'contiguous', 'masked'])
@pytest.mark.parametrize('layout,noted', [('token_contiguous', 1), ('row_major', 0)])
def test_calls_on_a_copy_of_the_scales_are_not_noted(monkeypatch, entry, layout, noted):
    """Large problems get a token-contiguous copy of row-major scales. What was launched then is no call that comes again, so noting it would
    be work on every call."""
    import yan_amd as yan
    from yan_amd.jit_kernels import gemm, m_grouped_gemm
    calls = []
    for module in (gemm, m_grouped_gemm):
        monkeypatch.setattr(module, 'remember_call', lambda call, *_: calls.append(call))
        monkeypatch.setattr(module, 'current_raw_stream', lambda: 0)
        monkeypatch.setattr(module, 'get_num_sms', lambda: 256)
    monkeypatch.setattr(gemm.jit_tuner, 'compile_and_tune', lambda **_: lambda *args: 0)
    m, n, k, groups = 4096, 7168, 7168, 4
    meta = lambda *shape, dtype: torch.empty(*shape, dtype=dtype, device='meta')
    code, scale, half = torch.float8_e4m3fn, torch.float32, torch.bfloat16
    lead = (groups, m // groups) if entry == 'masked' else (m, )
    scales = torch.ones(*lead, k // 128)
    lhs = meta(*lead, k, dtype=code), yan.get_col_major_tensor(scales) if layout == 'token_contiguous' else scales
    experts = () if entry == 'plain' else (groups, )
    rhs, out = (meta(*experts, n, k, dtype=code), meta(*experts, n // 128, k // 128, dtype=scale)), meta(*lead, n, dtype=half)
    if entry == 'plain':
        yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out)
    elif entry == 'contiguous':
        yan.m_grouped_gemm_fp8_fp8_bf16_nt_contiguous(lhs, rhs, out, meta(m, dtype=torch.int32))
    else:
        yan.m_grouped_gemm_fp8_fp8_bf16_nt_masked(lhs, rhs, out, meta(groups, dtype=torch.int32), m // groups)
    assert len(calls) == noted and all(call[2] is lhs[1] for call in calls)


def test_a_kernel_is_looked_at_once_for_all_sizes(monkeypatch):
    """Programs with ever new sizes note each of their calls: what is the kernel's own, its address and its kinds of arguments, is kept with it."""
    from yan_amd.jit.runtime import Runtime
    noted, looks = [], []
    cast = ctypes.cast
    monkeypatch.setattr(host_calls, '_host_calls', type('Module', (), {'remember': staticmethod(lambda *call: noted.append(call))}))
    monkeypatch.setattr(host_calls, 'repeat_call', lambda *_: False)
    monkeypatch.setattr(host_calls.ctypes, 'cast', lambda *a: (looks.append(a), cast(*a))[1])
    for name in ('YAN_SPLIT_K', 'YAN_TUNE_TILES'):
        monkeypatch.delenv(name, raising=False)
    monkeypatch.setattr(Runtime, 'is_path_valid', staticmethod(lambda path: True))
    runtime = Runtime('a_kernel')
    runtime._launch = ctypes.CFUNCTYPE(None)(lambda: None)
    runtime.args = (('a', torch.float32), ('alpha', float), ('workspace', torch.uint8), ('m', int), ('streamed', bool), ('b', torch.float32),
                    ('stream', torch.cuda.Stream))
    b, workspace = torch.nn.Parameter(torch.zeros(2)), torch.zeros(4, dtype=torch.uint8)
    for m in (1, 2, 3):
        a = torch.zeros(m)
        host_calls.remember_call((ENTRY, 1.0, a, b), 'a_kernel', runtime, (a, 1.0, workspace, m, True, b, 0), workspace)
        call, name, address, spec = noted.pop()
        assert call[2] is a and name == 'a_kernel' and address == cast(runtime._launch, ctypes.c_void_p).value
        assert spec == ((TENSOR, 0), (WORKSPACE, 0), (CONSTANT, m), (CONSTANT, 1), (TENSOR, 1), (STREAM, 0))
        host_calls.remember_call((ENTRY, 1.0, a), 'a_kernel', runtime, (a, 1.0, workspace, m, True, b, 0), workspace)
        assert not noted            # not every tensor of the launch is one of the call's
    assert len(looks) == 1
