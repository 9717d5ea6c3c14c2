"""Kernels and dispatch rules at the sizes where they can go wrong: edges of tiles, remainders, the ends of their ranges."""
import sys

import pytest
import torch

import oracle
import yan_amd as yan
import harness as testing
from yan_amd import jit

pytestmark = pytest.mark.gpu


def _announce(*what):
    print('[case]', *what, flush=True)
    sys.stdout.flush()


def _codes(t):
    return t.view(torch.uint8).cpu().numpy()


def _fp8_close(got, ref):
    """One bf16 step of rounding, plus what the matrix core drops inside a block of 128: up to 2^-15 of its largest product."""
    return bool(((got - ref).abs() <= ref.abs() * 2.0 ** -7 + 1e-4 * ref.abs().max()).all())


@pytest.mark.parametrize('rows,n,k,pad_blocks', testing.GROUPED_FOLLOW_GROUPS_CASES)
def test_contiguous_tiles_follow_the_groups(rows, n, k, pad_blocks):
    """fp8_gemm_contiguous_rows_kernel against the oracle, a workgroup per slot and eight workgroups walking them (same bits)."""
    from yan_amd.jit_kernels import m_grouped_gemm
    _announce('contiguous', rows, n, k, pad_blocks)
    (a8, sa), (b8, sb), out, idx = testing.make_grouped_contiguous_case(rows, n, k, seed=11, padding_blocks=pad_blocks)
    name, keys, arg_defs, code_template = testing.grouped_rows_on_device_plan(b8.size(0), n, k)
    kernel = jit.build(name, arg_defs, jit.generate(m_grouped_gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    ref = torch.from_numpy(oracle.m_grouped_gemm_contiguous_ref(_codes(a8), sa.numpy(), _codes(b8), sb.numpy(), idx.numpy(),
                                                                out_init=out.float().numpy()))
    a8d, sad, b8d, sbd, idxd = a8.cuda(), sa.cuda(), b8.cuda(), sb.cuda(), idx.cuda()
    results = []
    for cap in (256, 8):
        got = out.cuda()
        assert kernel(a8d, sad, b8d, sbd, got, idxd, a8.size(0), torch.cuda.current_stream(), cap, 0, sad.stride(0), sad.stride(1), 0, 0) == 0
        torch.cuda.synchronize()
        results.append(got.cpu())
    real = idx >= 0
    assert torch.equal(results[0], results[1])
    assert torch.equal(results[0][~real], out[~real])                   # padding blocks keep what they held
    assert _fp8_close(results[0][real].float(), ref[real])


@pytest.mark.parametrize('m,n,k', testing.FLOAT_SPLIT_K_SHAPES)
def test_float_split_k_matches_the_oracle_and_repeats(m, n, k):
    """gemm_cute_split_k through the entry: k that is no multiple of a k-tile or of the parts, last parts shorter than the
    others, tiles past n; alpha and beta, NaN in c with beta = 0; the same bits twice, counters back at zero."""
    from yan_amd.jit_kernels import simple_gemm, split_k
    _announce('fp32 split-K', m, n, k)
    name, keys, _ = simple_gemm.float_split_k_plan(m, n, k, 256)
    assert (keys['BLOCK_M'], keys['BLOCK_N'], keys['SPLIT_K']) == testing.FLOAT_SPLIT_K_SHAPES[(m, n, k)]
    a, b, c = testing.make_float_case(m, n, k, seed=13, device='cuda')
    start = torch.randn(m, n, generator=torch.Generator().manual_seed(14))
    ad, bd = a.double(), b.double()
    # every product and every sum of the at most k + 8 in a row rounds once, relative to the sum of magnitudes
    bound = (k + 8) * 2.0 ** -24 * (ad.abs() @ bd.abs().t() + start.abs().double().cuda()) * 2
    for alpha, beta in ((1.0, 0.0), (-0.5, 2.0)):
        results = []
        for _ in range(2):
            c.copy_(start if beta else torch.full_like(c, float('nan')))
            yan.gemm_float_nt(a, b, c, alpha=alpha, beta=beta)
            results.append(c.clone())
        want = alpha * (ad @ bd.t()) + (beta * start.double().cuda() if beta else 0.0)
        assert torch.equal(results[0], results[1])
        assert bool(((results[0].double() - want).abs() <= bound).all())
        assert ((results[0].double() - want).norm() / want.norm()).item() < 5e-6
    workspace, _ = split_k.split_k_workspace(c.device, torch.cuda.current_stream().cuda_stream)
    assert int(workspace[:split_k.SPLIT_K_COUNTER_BYTES].view(torch.int32).abs().sum()) == 0
