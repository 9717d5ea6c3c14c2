"""Repeated calls on the GPU (yan_amd/csrc/host_calls.cpp): every entry's native call against the Python way, captures and threads."""
import threading

import pytest
import torch

import harness as testing
import yan_amd as yan
from yan_amd.jit_kernels import bf16_gemm, fp8_cast, gemm, host_calls, m_grouped_gemm, simple_gemm

pytestmark = pytest.mark.gpu
MODULES = (bf16_gemm, fp8_cast, gemm, m_grouped_gemm, simple_gemm)


def _fp8(m, n, k, row_major=False):
    def make(seed):
        lhs, rhs, out = testing.make_fp8_case(m, n, k, seed=seed, device='cuda', gen_device='cuda', col_major_scales=not row_major)
        return (host_calls.FP8, *lhs, *rhs, out), lambda: yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out), [out]
    return make


def _bf16_fp8(m, n, k):
    def make(seed):
        _, rhs, out = testing.make_fp8_case(m, n, k, seed=seed, device='cuda', gen_device='cuda')
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).bfloat16().cuda()
        return (host_calls.CAST_FP8, x, *rhs, out), lambda: yan.gemm_bf16_fp8_bf16_nt(x, rhs, out), [out]
    return make


def _half(m, n, k, dtype):
    def make(seed):
        a, b, c = testing.make_bf16_case(m, n, k, seed=seed, dtype=dtype, device='cuda')
        bf16 = dtype == torch.bfloat16
        return (host_calls.BF16 if bf16 else host_calls.FP16, a, b, c), lambda: (yan.gemm_bf16_tn if bf16 else yan.gemm_fp16_tn)(a, b, c), [c]
    return make


def _float(m, n, k, alpha=1.0, beta=0.0):
    def make(seed):
        a, b, c = testing.make_float_case(m, n, k, seed=seed, device='cuda')
        start = torch.randn(m, n, generator=torch.Generator().manual_seed(seed)).cuda()

        def run():
            c.copy_(start)
            yan.gemm_float_nt(a, b, c, alpha, beta)
        return (host_calls.FLOAT, alpha, a, b, beta, c), run, [c, start]
    return make


def _contiguous(seed):
    lhs, rhs, out, idx = testing.make_grouped_contiguous_case((128, 128), 192, 256, seed=seed, device='cuda', padding_blocks=1)
    return (host_calls.CONTIGUOUS, *lhs, *rhs, out, idx), lambda: yan.m_grouped_gemm_fp8_fp8_bf16_nt_contiguous(lhs, rhs, out, idx), [out]


def _masked(expected_m):
    def make(seed):
        lhs, rhs, out, rows = testing.make_grouped_masked_case(2, 40, 192, 256, (40, 7), seed=seed, device='cuda')
        return ((host_calls.MASKED, *lhs, *rhs, out, rows, expected_m),
                lambda: yan.m_grouped_gemm_fp8_fp8_bf16_nt_masked(lhs, rhs, out, rows, expected_m), [out])
    return make


def _cast(kind, dtype):
    def make(seed):
        x = torch.randn(33 if kind == 'token' else 200, 384, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()
        entry = yan.per_token_cast_to_fp8 if kind == 'token' else yan.per_block_cast_to_fp8
        q = torch.zeros(x.shape, dtype=torch.float8_e4m3fn, device='cuda')
        scales = torch.zeros(x.size(0) if kind == 'token' else yan.ceil_div(x.size(0), 128), 3, device='cuda')
        number = host_calls.PER_TOKEN if kind == 'token' else host_calls.PER_BLOCK
        return (number, x, q, scales), lambda: [o.copy_(r) for o, r in zip((q, scales), entry(x))], [q, scales]
    return make


# an entry each, its kernels with and without a workspace, both layouts of scales
CALLS = {
    'fp8': _fp8(64, 256, 384), 'fp8 row-major': _fp8(64, 256, 384, True), 'fp8 split K': _fp8(40, 2112, 7168),
    'fp8 large row-major': _fp8(4096, 2048, 7168, True), 'fp8 weight streaming': _fp8(8, 2044, 1152),
    'bf16 to fp8': _bf16_fp8(64, 4096, 7168), 'bf16 to fp8, one kernel': _bf16_fp8(1, 2112, 7168),
    'bf16': _half(255, 132, 72, torch.bfloat16), 'bf16 split K': _half(100, 196, 3080, torch.bfloat16),
    'fp16': _half(8, 2044, 1152, torch.half), 'fp16 split K': _half(100, 196, 3080, torch.half),
    'fp32': _float(128, 64, 17, -0.5, 2.0), 'fp32 split K': _float(128, 64, 2050, 2.0, 1.0), 'fp32 on the bf16 cores': _float(4096, 4096, 1024),
    'contiguous': _contiguous, 'masked': _masked(40), 'masked, another hint': _masked(39),
    'quantise tokens': _cast('token', torch.bfloat16), 'quantise tokens fp32': _cast('token', torch.float32),
    'quantise weights': _cast('block', torch.bfloat16), 'quantise weights fp32': _cast('block', torch.float32),
}


def _bits(tensors):
    return [t.view(torch.uint8).clone() for t in tensors]


def _equal(tensors, bits):
    return all(torch.equal(t.view(torch.uint8), b) for t, b in zip(tensors, bits))


@pytest.fixture
def by_python(monkeypatch):
    """Runs something with the entries' way into native code shut."""
    def run(what):
        with monkeypatch.context() as m:
            for module in MODULES:
                m.setattr(module, 'repeat_call', lambda *_: False)
            what()
    return run


@pytest.mark.parametrize('name', CALLS)
def test_the_second_call_of_every_entry_is_native_and_right(name, by_python):
    """Other tensors than the first call's, all values other: the bits of the Python way."""
    print('[case] repeated', name, flush=True)
    host_calls._host_calls.forget()
    _, first, _ = CALLS[name](1)
    call, second, (out, *more) = CALLS[name](2)
    assert not host_calls.repeat_call(*call)
    first()
    by_python(second)
    want = _bits([out] + more)
    if name.startswith('fp32'):
        out.copy_(more[0])
    else:
        for t in (out, *more):
            t.fill_(-7.0)           # what the grouped outputs held before
    assert host_calls.repeat_call(*call)
    assert _equal([out] + more, want)


def test_hints_layouts_and_alignments_are_calls_of_their_own():
    """What a plan or a check looks at is part of what is compared: another hint of the masked entry, scales of a large problem that do not
    start on 16 bytes (they are copied, and their call is never a native one)."""
    host_calls._host_calls.forget()
    call, run, _ = _masked(40)(1)
    run()
    assert host_calls.repeat_call(*call) and not host_calls.repeat_call(*call[:-1], 39) and not host_calls.repeat_call(*call[:-1], 40.0)
    (_, q, scales, *rest), run, (out,) = _fp8(4096, 2048, 7168, True)(1)
    run()
    want = _bits([out])
    assert host_calls.repeat_call(host_calls.FP8, q, scales, *rest)
    moved = torch.empty(scales.numel() + 1, device='cuda')[1:].view_as(scales).copy_(scales)
    for _ in range(2):
        assert not host_calls.repeat_call(host_calls.FP8, q, moved, *rest)
        yan.gemm_fp8_fp8_bf16_nt((q, moved), tuple(rest[:2]), out)
        assert _equal([out], want)


def test_native_calls_without_a_workspace_are_captured():
    """A capture takes the launch as it is, on the capturing stream; replays follow what the tensors hold."""
    host_calls._host_calls.forget()
    call, run, (out,) = _fp8(64, 256, 384)(1)
    run()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert host_calls.repeat_call(*call)
    for seed in (2, 3, 2):
        (_, q, scales, w, ws, _), other, (want,) = _fp8(64, 256, 384)(seed)
        for old, new in zip(call[1:5], (q, scales, w, ws)):
            old.copy_(new)
        other()
        out.fill_(float('nan'))
        graph.replay()
        torch.cuda.synchronize()
        assert _equal([out], _bits([want]))


def test_threads_on_streams_of_their_own():
    """Native calls with a workspace from four threads at once, each on its stream and tensors: the bits that one thread gets."""
    print('[case] threads', flush=True)
    host_calls._host_calls.forget()
    cases = [CALLS[name](10 + i) for i, name in enumerate(('fp8 split K', 'bf16 split K', 'fp8 split K', 'bf16 to fp8'))]
    want = []
    for _, run, (out,) in cases:
        run()
        want += _bits([out])
    streams = [torch.cuda.Stream() for _ in cases]
    torch.cuda.synchronize()
    natively, wrong = [0] * 4, []

    def work(i):
        call, run, (out,) = cases[i]
        with torch.cuda.stream(streams[i]):
            for _ in range(50):
                out.fill_(float('nan'))
                if host_calls.repeat_call(*call):
                    natively[i] += 1
                else:
                    run()
                streams[i].synchronize()
                if not _equal([out], [want[i]]):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong and min(natively) >= 49


def test_streams_in_turn_stay_native():
    host_calls._host_calls.forget()
    call, run, (out,) = CALLS['fp8 split K'](1)
    run()
    want, side = _bits([out]), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    for _ in range(3):
        for stream in (torch.cuda.current_stream(), side):
            with torch.cuda.stream(stream):
                out.fill_(float('nan'))
                assert host_calls.repeat_call(*call)
                assert _equal([out], want)
            torch.cuda.synchronize()
