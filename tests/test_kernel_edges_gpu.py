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


def test_contiguous_tall_rows_of_the_last_round_run_flat():
    """On the whole chip, where only the row count decides: the bits of the same rows in one round (no row runs flat there)."""
    from yan_amd.jit_kernels import m_grouped_gemm
    rows, n, k = testing.GROUPED_LAST_ROUND_FLAT_CASE
    _announce('last round flat', rows, n, k)
    (a8, sa), (b8, sb), out, idx = testing.make_grouped_contiguous_case(rows, n, k, seed=25, device='cuda', gen_device='cuda')
    assert sum(rows) // 256 * (n // 256) == 264 and torch.cuda.get_device_properties(0).multi_processor_count == 256
    name, keys, arg_defs, code_template = testing.grouped_rows_on_device_plan(b8.size(0), n, k)
    kernel = jit.build(name, arg_defs, jit.generate(m_grouped_gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))

    def run(lo, hi):
        got, scales = out[lo:hi].clone(), yan.get_col_major_tensor(sa[lo:hi])
        assert kernel(a8[lo:hi], scales, b8, sb, got, idx[lo:hi], hi - lo, torch.cuda.current_stream(), 256, 0, scales.stride(0), scales.stride(1), 0, 0) == 0
        torch.cuda.synchronize()
        return got
    m = sum(rows)
    assert torch.equal(run(0, m), torch.cat([run(0, m // 2), run(m // 2, m)]))


@pytest.mark.parametrize('block_n,stages', testing.GROUPED_256_ROW_KEYS)
def test_contiguous_keys_that_name_a_tile_of_256_rows(block_n, stages):
    """Every width and depth such keys may hold, against the oracle, capped and not, with a row count that ends inside a block (the
    class takes one, the entries ask for whole blocks)."""
    from yan_amd.jit_kernels import m_grouped_gemm
    _announce('contiguous keys', block_n, stages)
    rows, n, k, pad_blocks = testing.GROUPED_256_ROW_KEYS_CASE
    (a8, sa), (b8, sb), out, idx = testing.make_grouped_contiguous_case(rows, n, k, seed=12, padding_blocks=pad_blocks)
    name, keys, arg_defs, code_template = testing.grouped_256_row_plan(block_n, stages, b8.size(0), n, k)
    kernel = jit.build(name, arg_defs, jit.generate(m_grouped_gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    ref = torch.from_numpy(oracle.m_grouped_gemm_contiguous_ref(_codes(a8), sa.numpy(), _codes(b8), sb.numpy(), idx.numpy(),
                                                                out_init=out.float().numpy()))
    a8d, sad, b8d, sbd, idxd = a8.cuda(), sa.cuda(), b8.cuda(), sb.cuda(), idx.cuda()
    for m in (a8.size(0), a8.size(0) - 60):
        results = []
        for cap in (256, 8):
            got = out.cuda()
            assert kernel(a8d, sad, b8d, sbd, got, idxd, m, torch.cuda.current_stream(), cap, 0, sad.stride(0), sad.stride(1), 0, 0) == 0
            torch.cuda.synchronize()
            results.append(got.cpu())
        written = (idx >= 0) & (torch.arange(a8.size(0)) < m)
        assert torch.equal(results[0], results[1])
        assert torch.equal(results[0][~written], out[~written])
        assert _fp8_close(results[0][written].float(), ref[written])


@pytest.mark.parametrize('tile,k', [(tile, k) for tile, depths in testing.FP8_WALK_CASES + testing.FP8_TWO_STAGE_LOOP_CASES for k in depths])
def test_fp8_walk_over_several_tiles_of_few_k_tiles(tile, k):
    m, n = testing.FP8_WALK_SIZES
    _announce('fp8 walk', tile, k)
    assert -(-m // tile[0]) * -(-n // tile[1]) > 2 * 8              # several tiles to a workgroup under the cap
    from yan_amd.jit_kernels import gemm
    (a8, sa), (b8, sb), out = testing.make_fp8_case(m, n, k, seed=16, device='cuda')
    name, keys, arg_defs, code_template = testing.fp8_explicit_tile_plan(*tile, n, k, 2)
    kernel = jit.build(name, arg_defs, jit.generate(gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    ref = torch.from_numpy(oracle.gemm_fp8_block_scaled_ref(_codes(a8), sa.cpu().numpy(), _codes(b8), sb.cpu().numpy()))
    sa_t, results = yan.get_col_major_tensor(sa), []
    for cap in (0, 8):
        out.fill_(float('nan'))
        assert kernel(a8, sa_t, b8, sb, out, m, torch.cuda.current_stream(), cap, 0) == 0
        torch.cuda.synchronize()
        results.append(out.cpu())
    assert torch.equal(results[0], results[1])
    assert _fp8_close(results[0].float(), ref)


@pytest.mark.parametrize('k', testing.MASKED_256_ROW_CASE[3])
def test_masked_layout_on_256_row_tiles_one_after_the_other(k):
    from yan_amd.jit_kernels import m_grouped_gemm
    m, n, masked, _ = testing.MASKED_256_ROW_CASE
    _announce('masked 256 rows', k)
    (a8, sa), (b8, sb), out, mm = testing.make_grouped_masked_case(len(masked), m, n, k, masked, seed=26)
    name, keys, arg_defs, code_template = testing.masked_256_row_plan(len(masked), n, k)
    kernel = jit.build(name, arg_defs, jit.generate(m_grouped_gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    ref = torch.from_numpy(oracle.m_grouped_gemm_masked_ref(_codes(a8), sa.numpy(), _codes(b8), sb.numpy(), mm.numpy(), out_init=out.float().numpy()))
    a8d, sad, b8d, sbd, mmd = a8.cuda(), sa.cuda(), b8.cuda(), sb.cuda(), mm.cuda()
    assert len(masked) * -(-m // 256) * -(-n // 256) > 2 * 8
    for expected_m in (m, 256):
        results = []
        for cap in (0, 8):
            got = out.cuda()
            assert kernel(a8d, sad, b8d, sbd, got, mmd, m, torch.cuda.current_stream(), cap, 0, sad.stride(1), sad.stride(2), sad.stride(0), expected_m) == 0
            torch.cuda.synchronize()
            results.append(got.cpu())
        assert torch.equal(results[0], results[1])
        for g, r in enumerate(masked):
            assert torch.equal(results[0][g, r:], out[g, r:]) and (r == 0 or _fp8_close(results[0][g, :r].float(), ref[g, :r]))


@pytest.mark.parametrize('col_major', [False, True])
@pytest.mark.parametrize('m,n,k', testing.CAPI_STREAMED_FP8_SIZES)
def test_library_streams_fp8_weights_to_the_same_bits(m, n, k, col_major):
    """All columns (weights streamed) against either half of them (not), with K split where the plan splits it and without."""
    from yan_amd import capi
    _announce('library, streamed fp8 weights', m, n, k, col_major)
    (a8, sa), (b8, sb), out = testing.make_fp8_case(m, n, k, seed=27, device='cuda', gen_device='cuda')
    if col_major:
        sa = yan.get_col_major_tensor(sa)
    ref = testing.dequant_lhs(a8, sa.contiguous()) @ testing.dequant_rhs(b8, sb).t()
    halves = []
    for lo, hi in ((0, n // 2), (n // 2, n)):
        halves.append(torch.full((m, hi - lo), float('nan'), dtype=torch.bfloat16, device='cuda'))
        assert capi.gemm_fp8_fp8_bf16_nt((a8, sa), (b8[lo:hi], sb[lo // 128:hi // 128]), halves[-1]) == 0
    out.fill_(float('nan'))
    assert capi.gemm_fp8_fp8_bf16_nt((a8, sa), (b8, sb), out) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, torch.cat(halves, dim=1)) and _fp8_close(out.float(), ref)
    out.fill_(float('nan'))
    assert capi.gemm_fp8_fp8_bf16_nt_split_k((a8, sa), (b8, sb), out, capi.split_k_workspace()) == 0
    torch.cuda.synchronize()
    assert _fp8_close(out.float(), ref)
    if capi.select_split_k(m, n, k, 256):           # the plan the entry compiles
        jit_out = torch.full_like(out, float('nan'))
        yan.gemm_fp8_fp8_bf16_nt((a8, sa), (b8, sb), jit_out)
        torch.cuda.synchronize()
        assert torch.equal(out, jit_out)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.half])
@pytest.mark.parametrize('m,n,k', testing.CAPI_STREAMED_DENSE_SIZES)
def test_library_spreads_and_streams_16_bit_weights_as_the_entry_does(m, n, k, dtype):
    from yan_amd import capi
    _announce('library, spread and streamed weights', m, n, k, dtype)
    a, b, c = testing.make_bf16_case(m, n, k, seed=28, dtype=dtype, device='cuda', gen_device='cuda')
    (yan.gemm_bf16_tn if dtype == torch.bfloat16 else yan.gemm_fp16_tn)(a, b, c)
    torch.cuda.synchronize()
    a64, b64 = a.double(), b.double()
    ref, magnitude = a64 @ b64.t(), a64.abs() @ b64.abs().t()
    # rounding to 8 or 11 bits, and fp32 sums of k products: k * 2^-24 of the sum of their magnitudes at the most
    bound = ref.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) + magnitude * (k * 2.0 ** -24)
    assert ((c.double() - ref).abs() <= bound).all()
    unsplit, split = torch.full_like(c, float('nan')), torch.full_like(c, float('nan'))
    assert (capi.gemm_bf16_tn if dtype == torch.bfloat16 else capi.gemm_fp16_tn)(a, b, unsplit) == 0
    assert capi.gemm_bf16_tn_split_k(a, b, split, capi.split_k_workspace()) == 0
    torch.cuda.synchronize()
    assert ((unsplit.double() - ref).abs() <= bound).all()
    assert torch.equal(split, c)                     # the same plan and kernel source


@pytest.mark.parametrize('k', testing.FP8_ODD_K_SIZES[2])
def test_fp8_few_k_tiles_an_odd_number_of_them_give_the_same_bits_walked_or_not(k):
    from yan_amd import capi
    from yan_amd.jit_kernels import gemm
    m, n, _ = testing.FP8_ODD_K_SIZES
    _announce('fp8 odd k-tiles', k)
    assert m * n * 2 > 64 << 20 >= m * n
    (a8, sa), (b8, sb), _ = testing.make_fp8_case(m, n, k, seed=24, device='cuda', gen_device='cuda')
    sa = yan.get_col_major_tensor(sa)
    outs = []
    for lo, hi in ((0, n), (0, n // 2), (n // 2, n)):
        name, keys, arg_defs, code_template = testing.fp8_explicit_tile_plan(*testing.FP8_ODD_K_TILE, hi - lo, k, 2)
        kernel = jit.build(name, arg_defs, jit.generate(gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
        outs.append(torch.full((m, hi - lo), float('nan'), dtype=torch.bfloat16, device='cuda'))
        assert kernel(a8, sa, b8[lo:hi], sb[lo // 128:hi // 128], outs[-1], m, torch.cuda.current_stream(), 0, 0) == 0
        torch.cuda.synchronize()
    assert torch.equal(outs[0], torch.cat(outs[1:], dim=1))
    # the library, whose kernel finds out when it runs
    via_lib = torch.full_like(outs[0], float('nan'))
    assert capi.gemm_fp8_fp8_bf16_nt((a8, sa), (b8, sb), via_lib) == 0
    torch.cuda.synchronize()
    assert torch.equal(via_lib, outs[0])
    half = torch.full_like(outs[1], float('nan'))
    assert capi.gemm_fp8_fp8_bf16_nt((a8, sa), (b8[:n // 2], sb[:n // 2 // 128]), half) == 0
    torch.cuda.synchronize()
    assert torch.equal(half, outs[1])
    rows = slice(0, m, 127)
    ref = testing.dequant_lhs(a8[rows], sa[rows].contiguous()) @ testing.dequant_rhs(b8, sb).t()
    assert _fp8_close(outs[0][rows].float(), ref)


@pytest.mark.parametrize('tile,k', [(tile, k) for tile, depths in testing.FP8_NARROW_TWO_STAGE_CASES for k in depths])
def test_fp8_two_stage_tiles_with_slabs_of_16_columns(tile, k):
    from yan_amd.jit_kernels import gemm
    m, n = testing.FP8_NARROW_TWO_STAGE_SIZES
    _announce('fp8 narrow', tile, k)
    (a8, sa), (b8, sb), out = testing.make_fp8_case(m, n, k, seed=23, device='cuda')
    name, keys, arg_defs, code_template = testing.fp8_explicit_tile_plan(*tile, n, k, 2)
    kernel = jit.build(name, arg_defs, jit.generate(gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    ref = torch.from_numpy(oracle.gemm_fp8_block_scaled_ref(_codes(a8), sa.cpu().numpy(), _codes(b8), sb.cpu().numpy()))
    sa_t, results = yan.get_col_major_tensor(sa), []
    for cap in (0, 8):
        out.fill_(float('nan'))
        assert kernel(a8, sa_t, b8, sb, out, m, torch.cuda.current_stream(), cap, 0) == 0
        torch.cuda.synchronize()
        results.append(out.cpu())
    assert torch.equal(results[0], results[1])
    assert _fp8_close(results[0].float(), ref)


@pytest.mark.parametrize('tile,k', [(tile, k) for tile, depths in testing.FP8_SHORT_K_TILES for k in depths])
def test_fp8_tiles_on_either_side_of_a_change_of_their_k_loop(tile, k):
    m, n = testing.FP8_SHORT_K_SIZES
    _announce('fp8 short k', tile, k)
    from yan_amd.jit_kernels import gemm
    (a8, sa), (b8, sb), out = testing.make_fp8_case(m, n, k, seed=15, device='cuda')
    name, keys, arg_defs, code_template = testing.fp8_explicit_tile_plan(*tile, n, k)
    kernel = jit.build(name, arg_defs, jit.generate(gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    ref = torch.from_numpy(oracle.gemm_fp8_block_scaled_ref(_codes(a8), sa.cpu().numpy(), _codes(b8), sb.cpu().numpy()))
    sa_t, results = yan.get_col_major_tensor(sa), []
    for cap in (0, 8):
        out.fill_(float('nan'))
        assert kernel(a8, sa_t, b8, sb, out, m, torch.cuda.current_stream(), cap, 0) == 0
        torch.cuda.synchronize()
        results.append(out.cpu())
    assert torch.equal(results[0], results[1])
    assert _fp8_close(results[0].float(), ref)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.half])
@pytest.mark.parametrize('tile', testing.DENSE_RAGGED_CAP_CASE[0])
def test_dense_ring_tiles_walked_with_ragged_rows_and_few_k_tiles(tile, dtype):
    _, (m, n), depths, cap = testing.DENSE_RAGGED_CAP_CASE
    for k in depths:
        _announce('dense ragged under a cap', tile, dtype, k)
        a, b, c = testing.make_bf16_case(m, n, k, seed=16, dtype=dtype, device='cuda')
        results = []
        for num_sms in (0, cap):
            name, keys, arg_defs, includes, code_template = testing.dense_tile_plan(tile, dtype, num_sms)
            kernel = jit.build(name, arg_defs, jit.generate(includes, arg_defs, jit.cpp_format(code_template, keys)))
            c.fill_(float('nan'))
            assert kernel(m, n, k, a, b, c, torch.cuda.current_stream()) == 0
            torch.cuda.synchronize()
            results.append(c.clone())
        ref = a.double().cpu() @ b.double().cpu().t()
        # one rounding of the result to its type, and of each of at most k + 8 sums in a row relative to the sum of magnitudes
        bound = ref.abs() * 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + (k + 8) * 2.0 ** -24 * (a.double().abs().cpu() @ b.double().abs().cpu().t())
        assert torch.equal(results[0], results[1])
        assert bool(((results[0].double().cpu() - ref).abs() <= bound).all())


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


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.half])
@pytest.mark.parametrize('tile,stages', testing.DENSE_LINE_WINDOW_TILES)
def test_rows_off_cache_lines_give_the_bits_of_the_smallest_tile(tile, stages, dtype):
    """Ring tiles that copy lines instead of rows' k-tiles (LineStager) against the 64 x 64 tile, which does not, and the product."""
    def kernel(which):
        name, keys, arg_defs, includes, code_template = testing.dense_tile_plan(which, dtype, 0)
        assert which != tile or keys['NUM_STAGES'] == stages
        return jit.build(name, arg_defs, jit.generate(includes, arg_defs, jit.cpp_format(code_template, keys)))
    lines, plain = kernel(tile), kernel((64, 64))
    for m, n, k, off_a, off_b in testing.DENSE_LINE_WINDOW_SHAPES:
        _announce('rows off lines', tile, dtype, m, n, k, off_a, off_b)
        g = torch.Generator().manual_seed(29)
        a_buf, b_buf = (torch.randn(rows * k + off + 64, generator=g).to(dtype).cuda() for rows, off in ((m, off_a), (n, off_b)))
        # what surrounds the operands must not get into a sum
        a_buf[:off_a], a_buf[off_a + m * k:], b_buf[:off_b], b_buf[off_b + n * k:] = (float('nan'),) * 4
        a, b = a_buf[off_a:off_a + m * k].view(m, k), b_buf[off_b:off_b + n * k].view(n, k)
        got, want = (torch.full((m + 2, n), 7.0, dtype=dtype, device='cuda') for _ in range(2))
        stream = torch.cuda.current_stream()
        assert lines(m, n, k, a, b, got[:m], stream) == 0 and plain(m, n, k, a, b, want[:m], stream) == 0
        assert torch.equal(got, want) and bool((got[m:] == 7.0).all())
        ad, bd = a.double(), b.double()
        ref = ad @ bd.t()
        # one rounding to the type, and at most k + 8 in a row of fp32 sums relative to the sum of magnitudes
        bound = ref.abs() * 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + (k + 8) * 2.0 ** -24 * (ad.abs() @ bd.abs().t())
        assert bool(((got[:m].double() - ref).abs() <= bound).all())


@pytest.mark.parametrize('cap', [0, testing.DENSE_LINE_WINDOW_CAP])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.half])
@pytest.mark.parametrize('tile', [tile for tile, _ in testing.DENSE_LINE_WINDOW_TILES])
def test_launches_that_copy_lines_give_the_bits_of_the_smallest_tile(tile, dtype, cap):
    """Sizes from which ring tiles copy lines, a workgroup per tile and fewer of them that walk the tiles."""
    def kernel(which, workgroups):
        name, keys, arg_defs, includes, code_template = testing.dense_tile_plan(which, dtype, workgroups)
        return jit.build(name, arg_defs, jit.generate(includes, arg_defs, jit.cpp_format(code_template, keys)))
    lines, plain = kernel(tile, cap), kernel((64, 64), 0)
    m, n = 11 * tile[0] - 5, 13 * tile[1] - 4
    for k, off_a, off_b in testing.DENSE_LINE_WINDOW_DEPTHS:
        _announce('launches that copy lines', tile, dtype, cap, k, off_a, off_b)
        g = torch.Generator(device='cuda').manual_seed(29)
        a_buf, b_buf = (torch.randn(rows * k + off + 64, generator=g, device='cuda').to(dtype) for rows, off in ((m, off_a), (n, off_b)))
        a_buf[:off_a], a_buf[off_a + m * k:], b_buf[:off_b], b_buf[off_b + n * k:] = (float('nan'),) * 4
        a, b = a_buf[off_a:off_a + m * k].view(m, k), b_buf[off_b:off_b + n * k].view(n, k)
        got, want = (torch.full((m + 2, n), 7.0, dtype=dtype, device='cuda') for _ in range(2))
        stream = torch.cuda.current_stream()
        assert lines(m, n, k, a, b, got[:m], stream) == 0 and plain(m, n, k, a, b, want[:m], stream) == 0
        assert torch.equal(got, want) and bool((got[m:] == 7.0).all())


@pytest.mark.parametrize('m,n,k', testing.WEIGHT_STREAM_SHAPES)
def test_weight_streaming_kernel_at_the_edges_of_its_tiles(m, n, k):
    """FP8 with both layouts of the activation scales, bf16 and fp16, through the entry points, against the product in float64; the
    rows behind the output stay untouched."""
    from yan_amd.jit_kernels import heuristics
    _announce('weight streaming', m, n, k)
    cus, atoms = yan.get_num_sms(), yan.ceil_div(m, 16)
    assert heuristics.get_weight_stream_fp8_config(m, n, k, cus) == heuristics.get_weight_stream_dense_config(m, n, k, cus) == atoms
    g = torch.Generator().manual_seed(31)
    x, w = (torch.randn(rows, k, generator=g) for rows in (m, n))

    def check(run, a, b, dtype, sum_error):
        out = torch.full((m + 2, n), 7.0, dtype=dtype, device='cuda')
        run(out[:m])
        assert bool((out[m:] == 7.0).all())
        ref = a @ b.t()
        # one rounding to the type, and an error per addition relative to the sum of magnitudes
        bound = ref.abs() * 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + (k + 8) * sum_error * (a.abs() @ b.abs().t())
        assert bool(((out[:m].double().cpu() - ref).abs() <= bound).all())

    for dtype, entry in ((torch.bfloat16, yan.gemm_bf16_tn), (torch.half, yan.gemm_fp16_tn)):
        a, b = x.to(dtype), w.to(dtype)
        check(lambda out: entry(a.cuda(), b.cuda(), out), a.double(), b.double(), dtype, 2.0 ** -24)
    wq, ws = yan.per_block_cast_to_fp8(w.bfloat16().cuda())
    b = wq.cpu().double() * ws.cpu().double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)
    for col_major in (True, False):
        xq, xs = yan.per_token_cast_to_fp8(x.bfloat16().cuda(), col_major_scales=col_major)
        # (the FP8 MFMA does not round its 128 products to nearest one by one: twice the error of a rounded sum)
        check(lambda out: yan.gemm_fp8_fp8_bf16_nt((xq, xs), (wq, ws), out), xq.cpu().double() * xs.cpu().double().repeat_interleave(128, 1), b,
              torch.bfloat16, 2.0 ** -23)


@pytest.mark.parametrize('m,n,k', testing.CAST_STREAM_SHAPES)
def test_activations_quantised_by_the_weight_streaming_kernel(m, n, k):
    """The bits of the quantiser and the FP8 entry one after the other, for ordinary rows, a row of zeros, an outlier, infinities and NaN; the
    rows behind the output stay untouched."""
    from yan_amd.jit_kernels import gemm as fp8_entry
    _announce('cast and weight streaming', m, n, k)
    assert fp8_entry.fp8_cast_stream_plan(m, n, k, yan.get_num_sms()) is not None
    g = torch.Generator().manual_seed(37)
    x = torch.randn(m, k, generator=g)
    x[0, 3], x[m // 2, k // 2:k // 2 + 64], x[m - 1, -1] = 3e4, 0.0, -2e-5
    w = yan.per_block_cast_to_fp8((torch.randn(n, k, generator=g) * k ** -0.5).bfloat16().cuda())
    for odd in (None, float('inf'), float('nan')):
        if odd is not None:
            x[m - 1, 7] = odd
        xd = x.bfloat16().cuda()
        two, one = (torch.full((m + 2, n), 7.0, dtype=torch.bfloat16, device='cuda') for _ in range(2))
        yan.gemm_fp8_fp8_bf16_nt(yan.per_token_cast_to_fp8(xd, col_major_scales=True), w, two[:m])
        yan.gemm_bf16_fp8_bf16_nt(xd, w, one[:m])
        assert bool((one[m:] == 7.0).all())
        assert torch.equal(one.isnan(), two.isnan()) and torch.equal(one.nan_to_num(), two.nan_to_num())


def _run_float_bf16x3(tile, parts, a, b, c, alpha=1.0, beta=0.0, lda=0, ldb=0):
    from yan_amd.jit_kernels import simple_gemm, split_k
    name, keys, arg_defs = testing.float_bf16x3_explicit_plan(tile, parts)
    kernel = jit.build(name, arg_defs, jit.generate(simple_gemm.bf16x3_includes, arg_defs, jit.cpp_format(simple_gemm.bf16x3_template, keys)))
    stream = torch.cuda.current_stream()
    args = (a.size(0), b.size(0), a.size(1), alpha, a, lda or a.size(0), b, ldb or b.size(0), beta, c, c.size(1), stream)
    if parts > 1:
        workspace, _ = split_k.split_k_workspace(c.device, stream.cuda_stream)
        args += (workspace, split_k.SPLIT_K_WORKSPACE_BYTES)
    assert kernel(*args) == 0


@pytest.mark.parametrize('tile,parts,shape', testing.FLOAT_BF16X3_CASES)
def test_float_on_the_bf16_cores_matches_the_product(tile, parts, shape):
    m, n, k = shape
    _announce('fp32 on bf16 cores', tile, parts, shape)
    a, b, _ = testing.make_float_case(m, n, k, seed=17, device='cuda')
    start = torch.randn(m + 1, n, generator=torch.Generator().manual_seed(18)).cuda()
    ad, bd = a.double(), b.double()
    # at most k + 16 roundings in a row, each relative to the sum of magnitudes
    bound = (k + 16) * 2.0 ** -24 * (ad.abs() @ bd.abs().t() + start[:m].abs().double()) * 2
    for alpha, beta in ((1.0, 0.0), (-0.5, 2.0)):
        results = []
        for _ in range(2):
            c = start.clone() if beta else torch.full_like(start, float('nan'))
            _run_float_bf16x3(tile, parts, a, b, c[:m], alpha, beta)
            results.append(c)
        want = alpha * (ad @ bd.t()) + (beta * start[:m].double() if beta else 0.0)
        assert torch.equal(results[0][:m], results[1][:m])
        assert bool(((results[0][:m].double() - want).abs() <= bound).all())
        assert torch.equal(results[0][m], start[m]) if beta else bool(results[0][m].isnan().all())


@pytest.mark.parametrize('tile,parts,shape', testing.FLOAT_BF16X3_CASES)
def test_what_lies_beside_the_operands_stays_out_of_the_bf16_cores(tile, parts, shape):
    """Leading dimensions beyond m and n with NaN or numbers that do not come apart behind the rows: the bits of operands without padding. (A
    tile that had gone to the fp32 cores for it would round otherwise.)"""
    m, n, k = shape
    _announce('fp32 on bf16 cores, padded', tile, parts, shape)
    a, b, want = testing.make_float_case(m, n, k, seed=37, device='cuda')
    _run_float_bf16x3(tile, parts, a, b, want)
    for junk in (float('nan'), 3e-36):
        wide_a, wide_b = (torch.full((k, rows + pad), junk, device='cuda') for rows, pad in ((m, 260), (n, 252)))
        wide_a[:, :m], wide_b[:, :n] = a.t(), b.t()
        got = torch.full((m + 1, n), 7.0, device='cuda')
        _run_float_bf16x3(tile, parts, wide_a.t()[:m], wide_b.t()[:n], got[:m], lda=m + 260, ldb=n + 252)
        assert torch.equal(got[:m], want) and bool((got[m:] == 7.0).all())


@pytest.mark.parametrize('tile,parts', [((256, 256), 1), ((128, 128), 5), ((128, 64), 7)])
def test_floats_that_do_not_come_apart_take_the_fp32_cores(tile, parts):
    """Numbers too small for three bf16, too large for the first of them, infinities, NaN and sums that leave the range give what the fp32
    matrix cores give; each kind alone, so that none hides behind another's second run of the tile."""
    m, n, k = 256, 256, 700
    big = torch.finfo(torch.float32).max
    for kind in ('tiny', 'subnormal', 'largest', 'infinity', 'nan', 'overflow'):
        _announce('fp32 on bf16 cores', tile, parts, kind)
        a, b, c = testing.make_float_case(m, n, k, seed=19, device='cuda')
        if kind == 'tiny':
            a[5] *= 2.0 ** -122
            b[:, ::2] *= 2.0 ** 60
        elif kind == 'subnormal':
            a[5, 3], a[5, 4:] = 2.0 ** -140, 0.0
            a[5, :3] = 0.0
            b[:, 3] = 2.0 ** 100
        elif kind == 'largest':
            a[5, 7] = big
            b[:, 7] = 2.0 ** -100
        elif kind == 'infinity':
            a[5, 7], b[9, 8] = float('inf'), float('-inf')
        elif kind == 'nan':
            a[5, 7] = float('nan')
        else:
            a[5, :200], b[9, :200] = 2.0 ** 65, 2.0 ** 63
        _run_float_bf16x3(tile, parts, a, b, c)
        ad, bd = a.double(), b.double()
        want = ad @ bd.t()
        beyond = want.isnan() | (want.abs() > big)
        assert bool(beyond[5].any()) == (kind in ('infinity', 'nan', 'overflow'))
        assert torch.equal(c.isnan(), want.isnan()) and torch.equal(c[beyond & ~want.isnan()].double(), want[beyond & ~want.isnan()].sign() * float('inf'))
        bound = (k + 16) * 2.0 ** -24 * (ad.abs() @ bd.abs().t()) * 2
        assert bool(((c.double() - want).abs() <= bound)[~beyond].all())


@pytest.mark.parametrize('tile,parts', [((256, 256), 1), ((128, 128), 5), ((128, 64), 7)])
def test_k_tiles_that_do_not_come_apart_are_added_once(tile, parts):
    """From the first such k-tile on the fp32 cores go on: in the first and the last, in neighbours, in one wave's step of a k-tile and in
    several, in either operand. One row (column) holds nothing but numbers that do not come apart, so that each of them is seen in the sum; the
    others see a k-tile that is left out or added twice."""
    m, n, k = 256, 256, 700
    for places in ([0], [k - 1], [15, 16], [300], [64, 150], [131, 132, 200], list(range(0, k, 97)), list(range(k))):
        for swapped in (False, True):
            _announce('k-tiles that do not come apart', tile, parts, places[:3], swapped)
            a, b, c = testing.make_float_case(m, n, k, seed=29, device='cuda')
            a[5] = 0.0
            a[5, places] = 2.0 ** -125 * (1.0 + 2.0 ** -20 * torch.arange(1, len(places) + 1, device='cuda'))
            b *= 2.0 ** 60
            if swapped:
                a, b = b, a
            results = []
            for _ in range(2):
                c.fill_(float('nan'))
                _run_float_bf16x3(tile, parts, a, b, c)
                results.append(c.clone())
            assert torch.equal(results[0], results[1])
            ad, bd = a.double(), b.double()
            bound = (k + 16) * 2.0 ** -24 * (ad.abs() @ bd.abs().t()) * 2
            assert bool(((c.double() - ad @ bd.t()).abs() <= bound).all())


def test_small_numbers_cost_no_second_run_of_their_tiles():
    """A number that does not come apart in every row: the entry takes about the time of the fp32 cores (measured 1.05 of it, 1.7 when such tiles
    were run on both), and about its own where it is the last k-tile's."""
    from yan_amd.jit_kernels import simple_gemm
    m, n, k = 4096, 4096, 1024
    _announce('time of small numbers', m, n, k)
    a, b, c = testing.make_float_case(m, n, k, seed=31, device='cuda')
    name, keys, arg_defs = simple_gemm.float_kernel_plan(m, n, 256)
    fp32 = jit.build(name, arg_defs, jit.generate(simple_gemm.includes, arg_defs, jit.cpp_format(simple_gemm.template, keys)))

    def microseconds(run):
        times = []
        for _ in range(12):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(5):
                run()
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end) * 200)
        return sorted(times)[3]

    entry = lambda: yan.gemm_float_nt(a, b, c)
    cores = microseconds(lambda: fp32(m, n, k, 1.0, a, m, b, n, 0.0, c, n, torch.cuda.current_stream()))
    usual = microseconds(entry)
    a[:, -1] = 3e-36
    late = microseconds(entry)
    a[:, 0] = 3e-36
    early = microseconds(entry)
    print(f'fp32 cores {cores:.1f} us, entry {usual:.1f}, small numbers in the last k-tile {late:.1f}, in the first {early:.1f}', flush=True)
    assert early < 1.3 * cores and late < 0.5 * (usual + cores)


@pytest.mark.parametrize('m,n,k', [(1024, 1024, 1024), (128, 2112, 7168), (640, 5120, 331)])
def test_float_on_the_bf16_cores_is_no_further_from_the_product(m, n, k):
    """Against 64 bits the error is no larger than on the fp32 matrix cores, with the same tile's parts of K or without."""
    from yan_amd.jit_kernels import simple_gemm
    _announce('fp32 error', m, n, k)
    name, keys, arg_defs = simple_gemm.float_kernel_plan(m, n, 256)
    fp32 = jit.build(name, arg_defs, jit.generate(simple_gemm.includes, arg_defs, jit.cpp_format(simple_gemm.template, keys)))
    for kind in ('normal', 'positive', 'wide'):
        a, b, c = testing.make_float_case(m, n, k, seed=23, device='cuda')
        if kind == 'positive':
            a, b = a.abs(), b.abs()
        elif kind == 'wide':
            a = a * torch.exp(3.0 * torch.randn(k, m, generator=torch.Generator().manual_seed(24)).cuda().t())
        want = a.double() @ b.double().t()
        assert fp32(m, n, k, 1.0, a, m, b, n, 0.0, c, n, torch.cuda.current_stream()) == 0
        before = ((c.double() - want).norm() / want.norm()).item()
        c.fill_(float('nan'))
        _run_float_bf16x3((128, 64), 1, a, b, c)
        after = ((c.double() - want).norm() / want.norm()).item()
        print(f'{kind}: {before:.2e} -> {after:.2e}', flush=True)
        assert after <= before


@pytest.mark.parametrize('m,n,k', testing.FLOAT_ERROR_SHAPES)
def test_float_entry_is_no_further_from_the_product_than_the_fp32_cores(m, n, k):
    """The entry's own plan on the bf16 cores against the plan that the fp32 cores would run, split or not: the error against 64 bits is no larger."""
    from yan_amd.jit_kernels import simple_gemm, split_k
    _announce('fp32 error of the entry', m, n, k)
    assert simple_gemm.float_bf16x3_plan(m, n, k, 256) is not None
    split = simple_gemm.float_split_k_plan(m, n, k, 256)
    name, keys, arg_defs = split or simple_gemm.float_kernel_plan(m, n, 256)
    code_template = simple_gemm.split_k_template if split else simple_gemm.template
    fp32 = jit.build(name, arg_defs, jit.generate(simple_gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    stream = torch.cuda.current_stream()
    for kind in ('normal', 'positive', 'wide'):
        a, b, c = testing.make_float_case(m, n, k, seed=41, device='cuda', gen_device='cuda')
        if kind == 'positive':
            a, b = a.abs(), b.abs()
        elif kind == 'wide':
            a = a * torch.exp(3.0 * torch.randn(k, m, generator=torch.Generator().manual_seed(42)).cuda().t())
        want = a.double() @ b.double().t()
        args = (m, n, k, 1.0, a, m, b, n, 0.0, c, n, stream)
        if split:
            workspace, _ = split_k.split_k_workspace(c.device, stream.cuda_stream)
            args += (workspace, split_k.SPLIT_K_WORKSPACE_BYTES)
        assert fp32(*args) == 0
        before = ((c.double() - want).norm() / want.norm()).item()
        c.fill_(float('nan'))
        yan.gemm_float_nt(a, b, c)
        after = ((c.double() - want).norm() / want.norm()).item()
        print(f'{kind}: {before:.2e} -> {after:.2e}', flush=True)
        assert after <= before


def _odd_floats(shape, dtype, seed):
    """Every kind of bit pattern: subnormals, huge values, zeros of both signs, and infinities and NaN here and there."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g) * torch.exp2(torch.randint(-130, 100, shape, generator=g).float())
    special = torch.tensor([float('inf'), float('-inf'), float('nan'), 0.0, -0.0])
    return torch.where(torch.rand(shape, generator=g) < 0.002, special[torch.randint(0, 5, shape, generator=g)], x).to(dtype)


def _groups_quantised(x, amax):
    """Codes and scales from each group's maximum, both quotients tensor by tensor (correctly rounded)."""
    factor = torch.full_like(amax, 448.0) / amax
    return x.float() * factor, amax / torch.full_like(amax, 448.0)


# below, at and past a workgroup's 32 rows; the last three on either side of where sources (32 MB) and codes (32 MB) are streamed
CAST_SHAPES = [(1, 128), (15, 384), (33, 128), (31, 4224), (65, 1152), (2341, 7168), (4682, 7168), (4097, 8192)]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('m,k', CAST_SHAPES)
def test_quantisers_on_odd_sizes_and_odd_values(m, k, dtype):
    """Both orders a workgroup takes its groups in and all three ways through the caches, against torch. A group with a NaN is
    scaled by the maximum of the others and a group with an infinity gets the scale infinity (codes there are NaN and 0)."""
    _announce('quantisers', m, k, dtype)
    x = _odd_floats((m, k), dtype, seed=m + k).cuda()
    tame = torch.where(torch.isnan(x.float()), torch.zeros((), device='cuda'), x.float().abs())
    amax = tame.view(m, k // 128, 128).amax(-1).clamp(min=1e-4)
    want, scales = _groups_quantised(x.view(m, k // 128, 128), amax.unsqueeze(-1))
    finite = (want.abs() <= 448.0).view(m, k)
    codes = want.view(m, k).to(torch.float8_e4m3fn).view(torch.uint8)
    for q, sc in (yan.per_token_cast_to_fp8(x), yan.per_token_cast_to_fp8(x, col_major_scales=True)):
        assert torch.equal(sc, scales.squeeze(-1))
        assert torch.equal(q.view(torch.uint8)[finite], codes[finite])
    block_amax = torch.nn.functional.pad(amax, (0, 0, 0, -m % 128)).view(-1, 128, k // 128).amax(1)
    want, _ = _groups_quantised(x, block_amax.repeat_interleave(128, 0)[:m].repeat_interleave(128, 1))
    q, sc = yan.per_block_cast_to_fp8(x)
    assert torch.equal(sc, block_amax / torch.full_like(block_amax, 448.0))
    finite = want.abs() <= 448.0
    assert torch.equal(q.view(torch.uint8)[finite], want.to(torch.float8_e4m3fn).view(torch.uint8)[finite])


def _streamed_weights_case(kind, tile, split_k):
    """The kernel on all columns (weights streamed) and on either half of them (not)."""
    dense = kind == 'dense'
    m, n, k = testing.STREAM_DENSE_SIZES if dense else testing.STREAM_FP8_SIZES
    outs = []
    if dense:
        a, b, c = testing.make_bf16_case(m, n, k, seed=17, device='cuda', gen_device='cuda')
    else:
        (a, sa), (b, sb), c = testing.make_fp8_case(m, n, k, seed=17, device='cuda', gen_device='cuda')
        sa = yan.get_col_major_tensor(sa)
    workspace = torch.zeros(16384 + (64 << 20), dtype=torch.uint8, device='cuda')
    stream = torch.cuda.current_stream()
    for lo, hi in ((0, n), (0, n // 2), (n // 2, n)):
        name, keys, arg_defs, includes, code_template = testing.stream_plans(kind, tile, split_k, hi - lo)
        kernel = jit.build(name, arg_defs, jit.generate(includes, arg_defs, jit.cpp_format(code_template, keys)))
        out = torch.full((m, hi - lo), float('nan'), dtype=torch.bfloat16, device='cuda')
        args = (m, hi - lo, k, a, b[lo:hi], out, stream) if dense else (a, sa, b[lo:hi], sb[lo // 128:hi // 128], out, m, stream, 0, 0)
        assert kernel(*args, *((workspace, workspace.numel()) if split_k > 1 else ())) == 0
        torch.cuda.synchronize()
        outs.append(out)
    return outs


@pytest.mark.parametrize('kind,tile,split_k', [('fp8', *c) for c in testing.STREAM_FP8_CASES] + [('dense', *c) for c in testing.STREAM_DENSE_CASES])
def test_streamed_weights_give_the_same_bits(kind, tile, split_k):
    _announce('streamed weights', kind, tile, split_k)
    whole, left, right = _streamed_weights_case(kind, tile, split_k)
    assert torch.equal(whole, torch.cat([left, right], dim=1))


@pytest.mark.parametrize('masked', [False, True])
def test_streamed_weights_of_groups_give_the_same_bits(masked):
    groups, rows, n, k = testing.STREAM_GROUPED_SIZES
    _announce('streamed weights of groups', masked)
    if masked:
        (a, sa), (b, sb), out, layout = testing.make_grouped_masked_case(groups, rows, n, k, (5, 64, 0, 1, 33, 64, 2, 17), seed=18, device='cuda', gen_device='cuda')
    else:
        (a, sa), (b, sb), out, layout = testing.make_grouped_contiguous_case((128, 7, 100, 1, 128, 64, 2, 90), n, k, seed=18, device='cuda', gen_device='cuda')

    def run(lo, hi):
        part = torch.full_like(out[..., lo:hi], -7.0, memory_format=torch.contiguous_format)
        rhs = b[:, lo:hi].contiguous(), sb[:, lo // 128:hi // 128].contiguous()
        if masked:
            yan.m_grouped_gemm_fp8_fp8_bf16_nt_masked((a, sa), rhs, part, layout, rows)
        else:
            yan.m_grouped_gemm_fp8_fp8_bf16_nt_contiguous((a, sa), rhs, part, layout)
        torch.cuda.synchronize()
        return part
    assert torch.equal(run(0, n), torch.cat([run(0, n // 2), run(n // 2, n)], dim=-1))


def _scale_layouts(scales):
    """The values of `scales` [..., rows, k/128] in the layouts a caller may hand over."""
    *lead, rows, blocks = scales.shape

    def row_pitch(extra, offset):
        buf = torch.full((*lead, rows, blocks + extra), float('nan'), device=scales.device).flatten()
        buf = torch.cat([torch.full((offset, ), float('nan'), device=scales.device), buf])[offset:].view(*lead, rows, blocks + extra)
        return buf[..., :blocks].copy_(scales)
    return {'row-major': scales.contiguous(), 'four apart': row_pitch(4, 0), 'one apart': row_pitch(1, 0), 'base off by one': row_pitch(0, 1),
            'base off by four': row_pitch(0, 4), 'every other': torch.stack([scales, scales], dim=-1).flatten(-2)[..., ::2]}


@pytest.mark.parametrize('tile,split_k,k', [(*t, k) for t in testing.SCALE_LAYOUT_TILES for k in testing.SCALE_LAYOUT_SIZES[2]])
def test_activation_scales_of_any_layout_give_the_same_bits(tile, split_k, k):
    from yan_amd.jit_kernels import gemm
    m, n, _ = testing.SCALE_LAYOUT_SIZES
    _announce('scale layouts', tile, split_k, k)
    (a8, sa), (b8, sb), out = testing.make_fp8_case(m, n, k, seed=19, device='cuda')
    name, keys, arg_defs, code_template = testing.strided_tile_plan(tile, split_k, n, k)
    kernel = jit.build(name, arg_defs, jit.generate(gemm.includes, arg_defs, jit.cpp_format(code_template, keys)))
    workspace = torch.zeros(16384 + 256 * 128 * 128 * 4, dtype=torch.uint8, device='cuda')

    def run(scales, cap=0):
        got = torch.full_like(out, float('nan'))
        split = (workspace, workspace.numel()) if split_k > 1 else ()
        assert kernel(a8, scales, b8, sb, got, m, torch.cuda.current_stream(), cap, 0, *split, *scales.stride()) == 0
        torch.cuda.synchronize()
        return got
    expected = run(yan.get_col_major_tensor(sa))
    ref = torch.from_numpy(oracle.gemm_fp8_block_scaled_ref(_codes(a8), sa.cpu().numpy(), _codes(b8), sb.cpu().numpy()))
    assert _fp8_close(expected.cpu().float(), ref)
    for layout, scales in _scale_layouts(sa).items():
        assert torch.equal(scales, sa), layout
        assert torch.equal(run(scales), expected), layout
    assert torch.equal(run(sa, 8), expected)
    same = sa[:1].expand(m, -1)
    assert torch.equal(run(same), run(yan.get_col_major_tensor(same.contiguous())))


@pytest.mark.parametrize('masked', [False, True])
def test_activation_scales_of_groups_of_any_layout_give_the_same_bits(masked):
    groups, rows, n, k = testing.STREAM_GROUPED_SIZES
    _announce('scale layouts of groups', masked)
    if masked:
        (a, sa), rhs, out, layout = testing.make_grouped_masked_case(groups, rows, n, k, (5, 64, 0, 1, 33, 64, 2, 17), seed=20, device='cuda', gen_device='cuda')
    else:
        (a, sa), rhs, out, layout = testing.make_grouped_contiguous_case((128, 7, 100, 1, 128, 64, 2, 90), n, k, seed=20, device='cuda', gen_device='cuda')

    def run(scales):
        got = torch.full_like(out, -7.0)
        if masked:
            yan.m_grouped_gemm_fp8_fp8_bf16_nt_masked((a, scales), rhs, got, layout, rows)
        else:
            yan.m_grouped_gemm_fp8_fp8_bf16_nt_contiguous((a, scales), rhs, got, layout)
        torch.cuda.synchronize()
        return got
    expected = run(yan.get_col_major_tensor(sa))
    for name, scales in _scale_layouts(sa).items():
        assert torch.equal(run(scales), expected), name


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.half])
@pytest.mark.parametrize('tile', testing.RAGGED_ROWS_CASE[0])
def test_output_rows_that_end_inside_a_16_byte_store(tile, dtype):
    """The bits of the same problem with four columns more, whose rows are whole 16-byte pieces, and nothing past the output."""
    _, m, columns, depths = testing.RAGGED_ROWS_CASE
    name, keys, arg_defs, includes, code_template = testing.dense_tile_plan(tile, dtype, 0)
    kernel = jit.build(name, arg_defs, jit.generate(includes, arg_defs, jit.cpp_format(code_template, keys)))
    stream = torch.cuda.current_stream()
    for k in depths:
        a, b, _ = testing.make_bf16_case(m, max(columns) + 4, k, seed=21, dtype=dtype, device='cuda')
        for n in columns:
            _announce('ragged rows', tile, dtype, n, k)
            whole = torch.full((m, n + 4), float('nan'), dtype=dtype, device='cuda')
            assert kernel(m, n + 4, k, a, b, whole, stream) == 0
            room = torch.full((m * n + 64, ), -7.0, dtype=dtype, device='cuda')
            assert kernel(m, n, k, a, b, room, stream) == 0
            torch.cuda.synchronize()
            assert torch.equal(room[:m * n].view(m, n), whole[:, :n])
            assert (room[m * n:] == -7.0).all()


@pytest.mark.parametrize('m,n,k', testing.ROTATED_SIZES)
@pytest.mark.parametrize('tile,split_k', testing.ROTATED_CASES)
def test_dense_tiles_that_start_at_different_places_along_k(tile, split_k, m, n, k):
    _announce('rotated', tile, split_k, m, n, k)
    a, b, c = testing.make_bf16_case(m, n, k, seed=22, device='cuda')
    name, keys, arg_defs, includes, code_template = testing.stream_plans('dense', tile, split_k, 0)
    kernel = jit.build(name, arg_defs, jit.generate(includes, arg_defs, jit.cpp_format(code_template, keys)))
    workspace = torch.zeros(16384 + 256 * 128 * 128 * 4, dtype=torch.uint8, device='cuda')
    results = []
    for _ in range(2):
        c.fill_(float('nan'))
        assert kernel(m, n, k, a, b, c, torch.cuda.current_stream(), *((workspace, workspace.numel()) if split_k > 1 else ())) == 0
        torch.cuda.synchronize()
        results.append(c.cpu())
    assert torch.equal(results[0], results[1])
    # bf16 rounding, and fp32 sums of k products: k * 2^-24 of the sum of their magnitudes at the most
    a64, b64 = a.double(), b.double()
    bound = (a64 @ b64.t()).abs() * 2.0 ** -8 + (a64.abs() @ b64.abs().t()) * (k * 2.0 ** -24)
    assert ((c.double() - a64 @ b64.t()).abs() <= bound).all()


def test_repeated_calls_are_made_natively_and_follow_what_changes(monkeypatch):
    """A call an entry has served before is made by the native host module; other sizes, strides and types, the compute-unit cap, the
    environment switches, another stream, a capture and wrong arguments still get what they ask for."""
    from yan_amd.jit_kernels import host_calls
    assert host_calls._host_calls is not None, 'yan_amd/csrc/build.py builds it'
    host_calls._host_calls.forget()
    m, n, k = 40, 2112, 7168                    # K is split: the call takes the stream's workspace
    _announce('repeated calls', m, n, k)
    cases = [testing.make_fp8_case(m, n, k, seed=s, device='cuda', col_major_scales=True) for s in (1, 2, 3)]
    refs = [testing.dequant_lhs(*lhs) @ testing.dequant_rhs(*rhs).t() for lhs, rhs, _ in cases]

    def right(out, ref):
        return float(yan.calc_diff(out.float(), ref)) < 1e-5

    def native(lhs, rhs, out):
        out.fill_(float('nan'))
        return host_calls.repeat_call(host_calls.FP8, *lhs, *rhs, out)

    lhs, rhs, out = cases[0]
    assert not native(lhs, rhs, out)
    yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out)
    for (lhs, rhs, out), ref in zip(cases, refs):       # other addresses, the same call
        assert native(lhs, rhs, out) and right(out, ref)
    lhs, rhs, out = cases[1]
    row_major = lhs[1].contiguous()
    assert row_major.stride() != lhs[1].stride() and not native((lhs[0], row_major), rhs, out)
    yan.gemm_fp8_fp8_bf16_nt((lhs[0], row_major), rhs, out)
    assert right(out, refs[1])
    assert not native((lhs[0][:39], lhs[1][:39]), rhs, out[:39]) and not native((lhs[0].cpu(), lhs[1]), rhs, out)
    with pytest.raises(AssertionError):
        yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out[:39])
    with pytest.raises(AssertionError):
        yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out.half())
    # what plans depend on
    full = yan.get_num_sms()
    try:
        yan.set_num_sms(64)
        assert not native(lhs, rhs, out)
        yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out)
        assert right(out, refs[1])
    finally:
        yan.set_num_sms(full)
    for name, value in (('YAN_SPLIT_K', '0'), ('YAN_TUNE_TILES', '1')):
        monkeypatch.setenv(name, value)
        assert not native(lhs, rhs, out)
        monkeypatch.delenv(name)
    assert native(lhs, rhs, out) and right(out, refs[1])
    # a stream of its own has a workspace of its own, and the first call on it goes round by Python; so does a capture
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert not native(lhs, rhs, out)
        yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out)
        assert native(lhs, rhs, out)
    torch.cuda.synchronize()
    assert right(out, refs[1])
    yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert not host_calls.repeat_call(host_calls.FP8, *lhs, *rhs, out)
        yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, out)
    for i in range(3):
        out.fill_(float('nan'))
        graph.replay()
        torch.cuda.synchronize()
        assert right(out, refs[1])
        yan.gemm_fp8_fp8_bf16_nt(lhs, rhs, cases[2][2])
    # one tensor in two places, then two; floats of the call
    x, y, c = testing.make_float_case(128, 128, 64, seed=4, device='cuda')
    for a, b in ((x, x), (x, y), (y, x)):
        for alpha, beta in ((1.0, 0.0), (-0.5, 2.0)):
            start = torch.ones_like(c)
            c.copy_(start)
            yan.gemm_float_nt(a, b, c, alpha, beta)
            assert torch.allclose(c.double(), alpha * (a.double() @ b.double().t()) + beta * start.double(), atol=1e-3)
            c.copy_(start)
            assert host_calls.repeat_call(host_calls.FLOAT, alpha, a, b, beta, c)
            assert torch.allclose(c.double(), alpha * (a.double() @ b.double().t()) + beta * start.double(), atol=1e-3)
