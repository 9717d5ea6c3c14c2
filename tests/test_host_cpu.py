"""Host-side logic that needs no device: helpers, tile heuristics, tuner selection rules, entry-point argument
checks (reference: yan/jit_kernels/utils.py:32-85, yan/jit_kernels/tuner.py:12-78, yan/jit_kernels/cute_gemm.py:21-30)."""
import os

import pytest
import torch

import yan_amd as yan
from yan_amd.jit_kernels import heuristics, tuner as tuner_mod, bf16_gemm, gemm, simple_gemm


def test_ceil_div_and_alignment():
    assert yan.ceil_div(7, 2) == 4 and yan.ceil_div(8, 2) == 4 and yan.ceil_div(0, 128) == 0 and yan.ceil_div(1, 128) == 1
    assert yan.get_m_alignment_for_contiguous_layout() == 128


def test_get_col_major_tensor():
    x = torch.arange(12, dtype=torch.float32).view(3, 4)
    y = yan.get_col_major_tensor(x)
    assert y.shape == x.shape and torch.equal(x, y) and y.stride() == (1, 3)
    assert yan.get_col_major_tensor(y).data_ptr() == y.data_ptr()          # already token-contiguous: untouched
    b = torch.arange(24, dtype=torch.float32).view(2, 3, 4)
    yb = yan.get_col_major_tensor(b)
    assert torch.equal(b, yb) and yb.stride(1) == 1 and yb.stride(2) == 3
    with pytest.raises(AssertionError):
        yan.get_col_major_tensor(torch.zeros(3))


def test_col_major_copies_of_matrices_are_those_of_batches():
    """A matrix is laid out as the only one of a batch is, whatever strides and sizes it comes with."""
    for rows in (0, 1, 2, 7):
        for cols in (0, 1, 3, 8):
            x = torch.randn(rows, 2 * cols + 1)
            for m in (x[:, :cols], x[:, ::2][:, :cols], torch.randn(cols, rows).t(), torch.randn(1, cols).expand(rows, cols), torch.randn(rows, cols)):
                got, want = yan.get_col_major_tensor(m), yan.get_col_major_tensor(m.unsqueeze(0)).squeeze(0)
                assert got.shape == want.shape and got.stride() == want.stride() and torch.equal(got, want)
                assert (got is m) == (m.stride() == (1, rows))


def test_tile_heuristics_fill_256_cus():
    # the headline FP8 shape: 256x256 tiles give 448 workgroups = 1.75 rounds
    assert heuristics.get_best_fp8_config(4096, 7168, 7168, 256) in ((256, 256), (256, 128), (128, 256))
    assert heuristics.get_best_dense_config(8192, 8192, 8192, 256) == (256, 256)
    # a skinny problem must not pick a tile that leaves most CUs idle
    bm, bn = heuristics.get_best_fp8_config(64, 4096, 7168, 256)
    assert yan.ceil_div(64, bm) * yan.ceil_div(4096, bn) >= 128
    # ... the decode shape runs the tiled kernel on 32 x 32 tiles (the 256 tiles of least operand traffic) with a deep ring of LDS stages, and up to 16 rows go
    # to the weight-streaming kernel (one workgroup per 16 weight rows) while those workgroups fit the chip at once
    assert heuristics.get_fp8_tile(64, 4096, 7168, 256) == (32, 32) and heuristics.get_fp8_num_stages(32, 32) == 12
    assert heuristics.get_fp8_tile(1, 4096, 7168, 256) == (16, 16) and heuristics.get_fp8_tile(16, 2048, 7168, 256) == (16, 16)
    assert heuristics.get_skinny_fp8_config(17, 4096, 7168, 256) == 0 and heuristics.get_skinny_fp8_config(16, 7168, 7168, 256) == 0
    assert heuristics.get_fp8_num_stages(256, 256) == 2 and heuristics.get_dense_num_stages(256, 256) == 2
    assert heuristics.get_dense_num_stages(64, 64) == 8 and heuristics.get_dense_num_stages(128, 256) == 3
    # tiny problems get the smallest tile
    assert heuristics.get_best_dense_config(64, 64, 64, 256) == (64, 64)
    # fp32: full tiles for large problems, K-split tiles (below 128 rows) when a 128-row tiling leaves CUs idle
    assert heuristics.get_best_float_config(8192, 8192, 256) == (256, 256)
    assert heuristics.get_best_float_config(4096, 7168, 256) == (128, 128)          # 1792 tiles: exactly 7 rounds
    assert heuristics.get_best_float_config(128, 2112, 256) == (32, 64)             # 33 tiles of 128 x 64 would use 33 CUs
    assert heuristics.get_best_float_config(128, 64, 256) == (32, 32)
    ranked = heuristics.rank_tiles(4096, 7168, 256, heuristics._FP8_TILES)
    assert ranked == sorted(ranked) and len(ranked) == len(heuristics._FP8_TILES)


def test_activation_scales_are_relaid_only_where_it_pays():
    """Large problems get token-contiguous activation scales (same values), small ones and scales that already are
    token-contiguous pass through untouched."""
    from yan_amd.jit_kernels.utils import scales_for_kernel, SCALE_RELAYOUT_MIN_FLOP
    rows = torch.arange(512 * 56, dtype=torch.float32).reshape(512, 56)
    assert scales_for_kernel(rows, SCALE_RELAYOUT_MIN_FLOP / 2) is rows
    big = scales_for_kernel(rows, SCALE_RELAYOUT_MIN_FLOP)
    assert big.stride() == (1, 512) and torch.equal(big, rows)
    assert scales_for_kernel(big, 1e15) is big
    one_block = rows[:, :1]
    assert scales_for_kernel(one_block, 1e15) is one_block
    batched = torch.arange(3 * 64 * 8, dtype=torch.float32).reshape(3, 64, 8)
    relaid = scales_for_kernel(batched, 1e15)
    assert relaid.stride() == (64 * 8, 1, 64) and torch.equal(relaid, batched)
    assert scales_for_kernel(relaid, 1e15) is relaid


def test_row_major_scales_stay_as_they_are_for_ring_tiles_up_to_k_8192():
    from yan_amd.jit_kernels.utils import scales_for_kernel
    ring = {'NUM_STAGES': 3, 'BLOCK_M': 128}
    for k_tiles, kept in ((32, True), (64, True), (68, False), (128, False), (30, False)):
        rows = torch.arange(128 * k_tiles, dtype=torch.float32).reshape(128, k_tiles)
        assert (scales_for_kernel(rows, 1e12, ring) is rows) == kept
        assert scales_for_kernel(rows, 1e12, {'NUM_STAGES': 2, 'BLOCK_M': 256}).stride() == (1, 128)
        assert torch.equal(scales_for_kernel(rows, 1e12, ring), rows)


def test_split_k_plans():
    """K is split when the unsplit tiles leave the chip short of work and K is long; every plan fits one round of
    workgroups and the workspace, leaves each part 14 k-tiles or more (24 of two), and the shapes of the GPU suite get the plans the
    suite expects (every ring tile, every factor)."""
    import harness
    plan = heuristics.get_split_k_fp8_config
    assert plan(64, 4096, 7168, 256) == (64, 64, 4) and plan(32, 2112, 7168, 256) == (32, 32, 3)
    assert plan(256, 7168, 7168, 256) == (128, 128, 2) and plan(128, 7168, 16384, 256) == (128, 128, 4)
    # short K, a weight matrix that takes as long to stream as to multiply, work for every compute unit, few rows
    assert plan(64, 7168, 2048, 256) is None and plan(64, 16384, 7168, 256) is None and plan(4096, 7168, 7168, 256) is None
    assert plan(16, 4096, 2048, 256) is None and plan(0, 4096, 7168, 256) is None
    assert plan(16, 4096, 7168, 256) == (32, 32, 2) and plan(1, 2112, 7168, 256) == (32, 32, 3)      # before the weight-streaming kernel
    for shape, expected in harness.FP8_SPLIT_K_PLAN_OF_SHAPE.items():
        assert plan(*shape, 256) == expected, shape
    assert {(bm, bn) for bm, bn, _ in harness.FP8_SPLIT_K_PLAN_OF_SHAPE.values()} == set(heuristics._FP8_SPLIT_K_TILE_US)
    assert {s for _, _, s in harness.FP8_SPLIT_K_PLAN_OF_SHAPE.values()} == set(heuristics.FP8_SPLIT_K_FACTORS)
    for m in (17, 33, 64, 100, 129, 256, 300, 512, 1024):
        for n in (196, 1536, 2112, 4096, 4100, 7168, 24576):
            for k in (1536, 3072, 3200, 4608, 7168, 16384):
                for cus in (256, 64, 8):
                    p = plan(m, n, k, cus)
                    if p is None:
                        continue
                    bm, bn, split = p
                    slots = yan.ceil_div(yan.ceil_div(m, bm) * yan.ceil_div(n, bn), 8) * 8
                    assert slots * split <= cus and yan.ceil_div(k // 128, split) >= (24 if split == 2 else 14)
                    assert gemm.SPLIT_K_COUNTER_BYTES + slots * split * bm * bn * 4 <= gemm.SPLIT_K_WORKSPACE_BYTES
                    assert slots * 8 * 4 <= gemm.SPLIT_K_COUNTER_BYTES
                    assert heuristics.get_fp8_num_stages(bm, bn) > 2          # a ring tile
    name, keys, defs, tmpl = gemm.fp8_split_k_plan(64, 4096, 7168, 256)
    assert name == 'gemm_fp8_fp8_bf16_nt_split_k' and keys['SPLIT_K'] == 4 and defs[-2:] == (('workspace', torch.uint8), ('workspace_bytes', int))
    assert 'run_split_k<4>' in yan.jit.cpp_format(tmpl, keys)
    strided = gemm.fp8_split_k_plan(64, 4096, 7168, 256, False)
    assert strided[0].endswith('_strided') and strided[2][-2:] == (('lhs_scales_stride_m', int), ('lhs_scales_stride_k', int))
    assert gemm.fp8_split_k_plan(4096, 7168, 7168, 256) is None


def test_dense_split_k_plans():
    """The dense GEMMs split K by the same rule with their own tile numbers: plans fit one round and the workspace, leave each
    part 16 k-tiles or more, and the shapes of the GPU suite get the plans the suite expects."""
    import harness
    plan = heuristics.get_split_k_dense_config
    assert plan(64, 4096, 7168, 256) == (64, 64, 4) and plan(256, 7168, 16384, 256) == (128, 128, 2)
    assert plan(256, 7168, 2048, 256) is None and plan(256, 24576, 1536, 256) is None and plan(8192, 8192, 8192, 256) is None
    assert plan(7, 4096, 7168, 256) is None and plan(16, 4096, 16384, 256) is None          # the one-atom weight-streaming kernel's
    assert plan(8, 4096, 7168, 256) == (64, 64, 4) and plan(17, 4096, 16384, 256) == (64, 64, 4)
    for shape, expected in harness.DENSE_SPLIT_K_PLAN_OF_SHAPE.items():
        assert plan(*shape, 256) == expected, shape
    assert {(bm, bn) for bm, bn, _ in harness.DENSE_SPLIT_K_PLAN_OF_SHAPE.values()} == set(heuristics._DENSE_SPLIT_K_EXTRA_US)
    assert {s for _, _, s in harness.DENSE_SPLIT_K_PLAN_OF_SHAPE.values()} == set(heuristics.DENSE_SPLIT_K_FACTORS)
    assert all((bm, bn) == (64, 64) for bm, bn, s in harness.DENSE_SPLIT_K_PLAN_OF_SHAPE.values() if s > 4)
    assert set(heuristics._DENSE_SPLIT_K_TILE_US) == {t for t in heuristics._DENSE_TILES if heuristics.get_dense_num_stages(*t) > 2}
    for m in (33, 64, 100, 129, 256, 300, 512, 1024):
        for n in (196, 1536, 2112, 4096, 4100, 7168, 24576):
            for k in (1536, 2048, 3080, 4608, 7168, 16384):
                for cus in (256, 64, 8):
                    p = plan(m, n, k, cus)
                    if p is None:
                        continue
                    bm, bn, split = p
                    slots = yan.ceil_div(yan.ceil_div(m, bm) * yan.ceil_div(n, bn), 8) * 8
                    assert slots * split <= cus and yan.ceil_div(yan.ceil_div(k, 64), split) >= 16
                    assert gemm.SPLIT_K_COUNTER_BYTES + slots * split * bm * bn * 4 <= gemm.SPLIT_K_WORKSPACE_BYTES
                    assert slots * 4 * 4 <= gemm.SPLIT_K_COUNTER_BYTES
    name, keys, defs = bf16_gemm.dense_split_k_plan(64, 4096, 7168, torch.half, 256)
    assert name == 'gemm_fp16_tn_split_k' and keys['SPLIT_K'] == 4 and defs[-2:] == (('workspace', torch.uint8), ('workspace_bytes', int))
    assert 'gemm_tn_split_k<BLOCK_M, BLOCK_N, kNumStages, kSplitK>' in bf16_gemm.split_k_template
    assert bf16_gemm.dense_split_k_plan(8192, 8192, 8192, torch.bfloat16, 256) is None


def test_fp8_shapes_of_the_gpu_suite_reach_every_tile_of_the_cost_table():
    import harness
    for shape, tile in harness.FP8_TILE_OF_SHAPE.items():
        assert shape in harness.FP8_TEST_SHAPES + harness.FP8_SIDE_SHAPES
        assert heuristics.get_fp8_tile(*shape, 256) == tile, shape
    assert set(harness.FP8_TILE_OF_SHAPE.values()) == set(heuristics._FP8_TILES)
    # two full rounds of 256 x 160 tiles beat 1.25 rounds of 256 x 256 tiles
    assert heuristics.get_best_fp8_config(4096, 5120, 5120, 256) == (256, 160)
    # the grouped layouts keep to widths of 64, 128 and 256
    assert heuristics.get_best_grouped_fp8_config(4096, 5120, 5120, 256, 1, 128, 4)[1] in (64, 128, 256)


def test_dense_shapes_of_the_gpu_suite_reach_every_tile_of_the_8_wave_kernel():
    """A change of the cost table must not silently take the 256 x {160, 192, 224} tiles, or the 192-wide ring tiles, out of the
    parity tests."""
    import harness
    for shape, tile in harness.DENSE_TILE_OF_SHAPE.items():
        assert shape in harness.DENSE_TEST_SHAPES
        assert heuristics.get_dense_tile(*shape, 256) == tile, shape
        if tile[1] != 16:
            assert heuristics.get_dense_num_stages(*tile) == (2 if tile[0] == 256 else {(128, 192): 4, (64, 192): 5}[tile])
    assert {t for t in harness.DENSE_TILE_OF_SHAPE.values()} == {(256, 160), (256, 192), (256, 224), (256, 256), (128, 192), (64, 192),
                                                                 (16, 16), (32, 16)}
    # shapes on which the launcher of the 256-row tiles takes the 4-wave kernel, every width among them, and shapes on which
    # it cannot
    for m, n, k in harness.DENSE_BOTH_KERNELS_SHAPES + [(8192, 8192, 8192)]:
        tile = heuristics.get_dense_tile(m, n, k, 256)
        assert tile[0] == 256 and tile[1] >= 160 and k % 64 == 0 and k >= 256 and n % 8 == 0
    assert {heuristics.get_dense_tile(*shape, 256)[1] for shape in harness.DENSE_BOTH_KERNELS_SHAPES} == {160, 192, 224, 256}
    assert 1000 % 64 != 0 and 5004 % 8 != 0 and 520 % 64 != 0 and 264 % 64 != 0 and 72 < 256
    # the weight-streaming kernel: one round of workgroups, whole K blocks, two atoms only on long K
    assert heuristics.get_skinny_dense_config(16, 4096, 7168, 256) == 1 and heuristics.get_skinny_dense_config(16, 4112, 7168, 256) == 0
    assert heuristics.get_skinny_dense_config(16, 4096, 7176, 256) == 0 and heuristics.get_skinny_dense_config(33, 4096, 7168, 256) == 0
    assert heuristics.get_skinny_dense_config(32, 4096, 1024, 256) == 0 and heuristics.get_skinny_dense_config(32, 4096, 2048, 256) == 2
    assert heuristics.get_skinny_dense_config(16, 1024, 7168, 64) == 1 and heuristics.get_skinny_dense_config(16, 2048, 7168, 64) == 0


def test_kernel_plans_keep_reference_keys_and_argument_order():
    name, keys, defs = bf16_gemm.dense_kernel_plan(4096, 7168, 2048, torch.bfloat16, 256)
    assert name == 'gemm_bf16_tn' and sorted(keys) == ['BLOCK_M', 'BLOCK_N', 'NUM_SMS', 'NUM_STAGES'] and keys['NUM_SMS'] == 0
    assert bf16_gemm.dense_kernel_plan(4096, 7168, 2048, torch.bfloat16, 64, 64)[1]['NUM_SMS'] == 64
    assert [d[0] for d in defs] == ['m', 'n', 'k', 'A', 'B', 'C', 'stream']
    assert bf16_gemm.dense_kernel_plan(4096, 7168, 2048, torch.half, 256)[0] == 'gemm_fp16_tn'
    name, keys, defs, smem, _ = gemm.fp8_kernel_plan(4096, 7168, 7168, 256)
    assert name == 'gemm_fp8_fp8_bf16_nt'
    assert sorted(keys) == ['BLOCK_M', 'BLOCK_N', 'K', 'N', 'NUM_STAGES', 'NUM_TMA_MULTICAST']
    # the reference's nine run-time names, exactly (yan/jit_kernels/gemm.py:23-30), for token-contiguous activation scales
    assert [d[0] for d in defs] == ['lhs', 'lhs_scales', 'rhs', 'rhs_scales', 'out', 'm', 'stream', 'num_sms', 'smem_size']
    assert defs is gemm.arg_defs and gemm.fp8_kernel_plan(4096, 7168, 7168, 256)[4] is gemm.template
    # any other strided layout: the same, plus the two strides
    strided = gemm.fp8_kernel_plan(4096, 7168, 7168, 256, False)
    assert [d[0] for d in strided[2]] == [d[0] for d in defs] + ['lhs_scales_stride_m', 'lhs_scales_stride_k'] and strided[1] == keys
    assert strided[0] == 'gemm_fp8_fp8_bf16_nt_strided'           # its own name: the tuner memoises per (name, keys)
    name, fkeys, defs = simple_gemm.float_kernel_plan(4096, 7168, 256)
    assert name == 'gemm_float_nt' and sorted(fkeys) == ['BLOCK_M', 'BLOCK_N']
    assert [d[0] for d in defs] == ['m', 'n', 'k', 'alpha', 'A', 'ldA', 'B', 'ldB', 'beta', 'C', 'ldC', 'stream']
    assert keys['N'] == 7168 and keys['K'] == 7168 and smem == 2 * (keys['BLOCK_M'] + keys['BLOCK_N']) * 128 <= 160 * 1024


def test_entry_points_reject_bad_arguments_before_touching_a_device():
    a, b = torch.zeros(8, 16, dtype=torch.bfloat16), torch.zeros(4, 16, dtype=torch.bfloat16)
    with pytest.raises(AssertionError):
        yan.gemm_bf16_tn(a, b, torch.zeros(8, 8, dtype=torch.bfloat16))          # n mismatch
    with pytest.raises(AssertionError):
        yan.gemm_bf16_tn(a.half(), b, torch.zeros(8, 4, dtype=torch.bfloat16))   # dtype mismatch
    with pytest.raises(AssertionError):
        yan.gemm_fp16_tn(a, b, torch.zeros(8, 4, dtype=torch.bfloat16))
    # empty problems return before any device call
    yan.gemm_bf16_tn(torch.zeros(0, 16, dtype=torch.bfloat16), b, torch.zeros(0, 4, dtype=torch.bfloat16))
    yan.gemm_fp16_tn(torch.zeros(8, 16, dtype=torch.half), torch.zeros(0, 16, dtype=torch.half), torch.zeros(8, 0, dtype=torch.half))
    # fp32 GEMM (yan/jit_kernels/simple_gemm.py:25-32): m % 128, n % 64, dtypes, shapes; operands M- / N-contiguous
    x, y = yan.get_col_major_tensor(torch.zeros(128, 16)), yan.get_col_major_tensor(torch.zeros(64, 16))
    with pytest.raises(AssertionError):
        yan.gemm_float_nt(x[:100], y, torch.zeros(100, 64))
    with pytest.raises(AssertionError):
        yan.gemm_float_nt(x, y[:32], torch.zeros(128, 32))
    with pytest.raises(AssertionError):
        yan.gemm_float_nt(x, y, torch.zeros(128, 128))
    with pytest.raises(AssertionError):
        yan.gemm_float_nt(x.double(), y, torch.zeros(128, 64))
    with pytest.raises(AssertionError):     # row-major operands would be read as their transposes
        yan.gemm_float_nt(torch.zeros(128, 16), y, torch.zeros(128, 64))
    yan.gemm_float_nt(yan.get_col_major_tensor(torch.zeros(0, 16)), y, torch.zeros(0, 64))
    q = torch.zeros(0, 128, dtype=torch.float8_e4m3fn)
    w = torch.zeros(128, 128, dtype=torch.float8_e4m3fn)
    yan.gemm_fp8_fp8_bf16_nt((q, torch.zeros(0, 1)), (w, torch.ones(1, 1)), torch.zeros(0, 128, dtype=torch.bfloat16))
    with pytest.raises(AssertionError):     # k not a multiple of the 128-deep scale block
        yan.gemm_fp8_fp8_bf16_nt((torch.zeros(4, 64, dtype=torch.float8_e4m3fn), torch.zeros(4, 1)),
                                 (torch.zeros(128, 64, dtype=torch.float8_e4m3fn), torch.ones(1, 1)),
                                 torch.zeros(4, 128, dtype=torch.bfloat16))
    with pytest.raises(AssertionError):     # wrong scale-table shape
        yan.gemm_fp8_fp8_bf16_nt((torch.zeros(4, 128, dtype=torch.float8_e4m3fn), torch.zeros(4, 2)),
                                 (w, torch.ones(1, 1)), torch.zeros(4, 128, dtype=torch.bfloat16))


class _FakeRuntime:
    def __init__(self, tag, rc=0):
        self.tag, self.rc, self.calls = tag, rc, 0

    def __call__(self, *args):
        self.calls += 1
        return self.rc


def test_tuner_memoises_skips_illegal_and_keeps_the_fastest(monkeypatch):
    built = []
    times = {'a': 3.0, 'b': 1.0, 'c': 2.0, 'bad': 0.1}

    def fake_build(name, arg_defs, code):
        tag = code.split('TAG=')[1].split(';')[0]
        rt = _FakeRuntime(tag, rc=5 if tag == 'bad' else 0)
        built.append(rt)
        return rt

    monkeypatch.setattr(tuner_mod, 'build', fake_build)
    monkeypatch.setattr(tuner_mod, '_time_candidate', lambda rt, args: times[rt.tag])
    t = tuner_mod.JITTuner()
    kw = dict(includes=(), arg_defs=(('n', int),), template='\nint TAG={T}; int k={KEY};\n', args=(1,))
    space = ({'T': 'a'}, {'T': 'bad'}, {'T': 'b'}, {'T': 'c'})
    best = t.compile_and_tune(name='op', keys={'KEY': 1}, space=space, **kw)
    assert best.tag == 'b' and len(built) == 4
    assert [r.calls for r in built] == [1, 1, 1, 1]              # one validity run each; the illegal one is not timed
    # memo hit: same name and keys (in any order) -> no new build
    assert t.compile_and_tune(name='op', keys={'KEY': 1}, space=space, **kw) is best and len(built) == 4
    # different keys -> new entry; empty space -> exactly one build, not run, time 0
    one = t.compile_and_tune(name='op', keys={'KEY': 2, 'T': 'c'}, space=(), **kw)
    assert one.tag == 'c' and one.calls == 0 and len(built) == 5
    # every candidate illegal -> assertion
    with pytest.raises(AssertionError, match='Failed to tune'):
        t.compile_and_tune(name='op2', keys={'KEY': 3}, space=({'T': 'bad'}, {'T': 'bad'}), **kw)


def test_reference_package_name_is_an_alias():
    """Code written against the reference imports `yan` (tests/test_cute.py:5-6 there); here that name resolves to
    this package, with the names that test uses."""
    import yan as by_reference_name
    assert by_reference_name is yan
    for name in ('gemm_fp16_tn', 'bench_kineto', 'get_col_major_tensor', 'calc_diff', 'jit', 'jit_kernels', 'gemm'):
        assert hasattr(by_reference_name, name), name
    assert callable(by_reference_name.jit_kernels.cute_gemm_accuracy_test)


def test_tile_scheduler_visits_every_tile_once_and_walks_cover_every_slot(tmp_path, repo_root):
    """XcdTileScheduler::tile_of and capped_grid are __host__ __device__: the checks live in tests/scheduler_host.cpp,
    compiled for the host only."""
    import subprocess
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir
    exe = tmp_path / 'scheduler_host'
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-host-only', '-std=c++20', '-O1', f'-I{get_jit_include_dir()}',
                           os.path.join(repo_root, 'tests', 'scheduler_host.cpp'), '-o', str(exe)])
    done = subprocess.run([str(exe)], stdout=subprocess.PIPE, universal_newlines=True)
    assert done.returncode == 0 and done.stdout.startswith('ok '), done.stdout
    assert int(done.stdout.split()[1]) > 400


def test_weights_are_streamed_where_that_measured_faster():
    """Shapes that the split-K plan or the tiles measured faster on go there, neighbours that they did not stay with the weight-streaming kernel."""
    dense = {(14, 4428, 15360): 0, (16, 4428, 7168): 1, (17, 4736, 8832): 0, (18, 5888, 8832): 2, (6, 7992, 15872): 0, (3, 7936, 9984): 1,
             (4, 12288, 8192): 0, (4, 12288, 6144): 1, (1, 15116, 4608): 0, (4, 14080, 3072): 1, (30, 13888, 1408): 0, (32, 14336, 2048): 2, (32, 16384, 256): 2,
             (48, 4096, 4480): 0, (24, 4096, 7168): 2, (63, 7872, 2688): 0, (58, 7168, 1792): 4, (16, 1472, 15104): 1}
    fp8 = {(25, 1856, 9728): 0, (25, 1856, 7168): 2, (10, 13184, 11264): 0, (2, 13184, 11264): 1, (32, 16384, 16384): 2}
    for (m, n, k), atoms in dense.items():
        assert heuristics.get_weight_stream_dense_config(m, n, k, 256) == atoms, (m, n, k)
    for (m, n, k), atoms in fp8.items():
        assert heuristics.get_weight_stream_fp8_config(m, n, k, 256) == atoms, (m, n, k)


def test_launches_copy_lines_only_where_that_pays(tmp_path):
    """copies_whole_lines: rows off lines, by K or by where both operands start; half of the chip at work; enough k-tiles for the tile."""
    import subprocess
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir
    source, exe = tmp_path / 'rule.cpp', tmp_path / 'rule'
    source.write_text("""
#include "gemm/bf16_gemm.hpp"
#include <cstdio>
int main() {
    int block_m, block_n, parts, groups, k;
    long a, b;
    while (std::scanf("%d %d %d %d %d %ld %ld", &block_m, &block_n, &parts, &groups, &k, &a, &b) == 7)
        std::printf("%d ", int(yan::copies_whole_lines(block_m, block_n, parts, groups, k, reinterpret_cast<void*>(a), reinterpret_cast<void*>(b))));
}
""")
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-host-only', '-std=c++20', '-O1', '-w', f'-I{get_jit_include_dir()}', str(source),
                           '-o', str(exe)])
    cases = {
        # the tile, parts of K, workgroups, K, where the operands start
        (64, 128, 1, 136, 600, 4096, 4096): 0, (64, 128, 1, 136, 1272, 4096, 4096): 1, (64, 128, 1, 250, 968, 4096, 4096): 1, (64, 128, 1, 250, 952, 4096, 4096): 0,
        (64, 128, 1, 120, 4104, 4096, 4096): 0, (64, 192, 1, 190, 520, 4096, 4096): 1, (64, 192, 1, 190, 504, 4096, 4096): 0,
        (128, 128, 1, 255, 600, 4096, 4096): 0, (128, 128, 1, 255, 712, 4096, 4096): 1, (128, 192, 1, 230, 600, 4096, 4096): 0,
        (128, 192, 1, 200, 600, 4096, 4096): 1, (64, 128, 3, 216, 4104, 4096, 4096): 1, (64, 128, 4, 216, 4104, 4096, 4096): 1, (64, 128, 4, 216, 3960, 4096, 4096): 0,
        (64, 128, 4, 216, 4040, 4096, 4096): 1,
        (128, 192, 1, 200, 4096, 4096, 4096): 0, (128, 192, 1, 200, 4096, 4112, 4096): 0, (128, 192, 1, 200, 4096, 4096, 4112): 0,
        (128, 192, 1, 200, 4096, 4112, 4128): 1, (128, 192, 1, 200, 4128, 4096, 4096): 0,
    }
    done = subprocess.run([str(exe)], input='\n'.join(' '.join(map(str, c)) for c in cases), stdout=subprocess.PIPE, universal_newlines=True, check=True)
    assert dict(zip(cases, map(int, done.stdout.split()))) == cases


@pytest.mark.parametrize('shape,dtype_name', [((8192, 8192, 8192), 'bfloat16'), ((4096, 5120, 5120), 'bfloat16'), ((8192, 8192, 8192), 'half')])
def test_tied_accumulators_of_the_8_wave_kernel_stay_where_the_mfmas_left_them(tmp_path, shape, dtype_name):
    """The 8-wave dense kernel writes its MFMAs as asm statements whose destination is their own addend. The compiler does
    not know how long such an instruction takes, so nothing but MFMAs may touch an accumulator register between the first
    and the last MFMA of the main loop (a compiler-made copy right behind an MFMA would read a sum that is not there yet),
    and what reads them first afterwards must sit behind the wait states written in the source. Checked on the generated
    code: compiled for the device only, no GPU needed."""
    import re
    import subprocess
    from yan_amd.jit import cpp_format, generate
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    from yan_amd.jit_kernels import bf16_gemm
    dtype = getattr(torch, dtype_name)
    _, keys, arg_defs = bf16_gemm.dense_kernel_plan(*shape, dtype, 256, 0)
    assert keys['BLOCK_M'] == 256 and keys['NUM_STAGES'] == 2             # the 8-wave kernel
    src, asm = tmp_path / 'kernel.cu', tmp_path / 'kernel.s'
    src.write_text(generate(bf16_gemm.includes, arg_defs, cpp_format(bf16_gemm.template, keys)))
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-device-only', '-S', '-std=c++20', '-O3',
                           f'--offload-arch={get_offload_arch()}', '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
                           f'-I{get_jit_include_dir()}', str(src), '-o', str(asm)])
    text = asm.read_text()
    assert re.search(r'\.private_segment_fixed_size:\s+0\b', text), 'the kernel spills'
    # instructions and labels of the kernel, in text order
    lines = [line.split(';')[0].strip() for line in text.split('\n')]
    lines = [line for line in lines if line and (line.endswith(':') or not line.startswith(('.', '//')))]

    def regs(operand_text):
        found = set()
        for lo, hi in re.findall(r'\bv\[(\d+):(\d+)\]', operand_text):
            found.update(range(int(lo), int(hi) + 1))
        found.update(int(r) for r in re.findall(r'\bv(\d+)\b', operand_text))
        return found

    mfma = re.compile(r'^v_mfma_f32_16x16x32_(?:bf16|f16) (v\[\d+:\d+\]), (v\[\d+:\d+\]), (v\[\d+:\d+\]), (v\[\d+:\d+\])')
    where = [i for i, line in enumerate(lines) if mfma.match(line)]
    assert len(where) >= 2 * 2 * keys['BLOCK_N'] // 32 * 4          # at least the steps of two k-tiles
    acc = set()
    for i in where:
        dst, a, b, c = mfma.match(lines[i]).groups()
        assert dst == c, lines[i]                                    # accumulates in place
        acc |= regs(dst)
    assert len(acc) == 256 * keys['BLOCK_N'] // 512                  # one register per output of the wave's slab
    for i in where:
        _, a, b, _ = mfma.match(lines[i]).groups()
        assert not (regs(a) | regs(b)) & acc, lines[i]

    def mfma_in_flight_before(i):
        """An MFMA less than 20 instructions up the straight-line path that ends at instruction i, with no `s_nop 15`
        pair between; a path stops at a label whose predecessor in the text ends with an unconditional branch."""
        nops = 0
        for back in range(1, 21):
            line = lines[i - back]
            if line.endswith(':'):
                if lines[i - back - 1].startswith('s_branch'):
                    return False
                continue
            if line == 's_nop 15':
                nops += 1
            if mfma.match(line):
                return nops < 2
        return False
    for i in range(where[0], len(lines)):
        line = lines[i]
        if mfma.match(line) or line.endswith(':') or line.startswith('s_') or not regs(line) & acc:
            continue
        assert not mfma_in_flight_before(i), f'{line} touches an accumulator right behind an MFMA'
    # and the epilogue's first read of a sum sits behind the wait states written in the source
    after = lines[where[-1] + 1:]
    first_use = next(i for i, line in enumerate(after) if not line.endswith(':') and not line.startswith('s_') and regs(line) & acc)
    assert sum(1 for line in after[:first_use] if line == 's_nop 15') >= 2, 'the sums are read before the last MFMAs have retired'


@pytest.mark.parametrize('dtype_name', ['bfloat16', 'half'])
def test_the_4_wave_dense_kernel_keeps_its_sums_in_place_and_one_instruction_behind_each_mfma(tmp_path, dtype_name):
    """The 4-wave kernel of the 256 x 256 tile has one wave per SIMD: a spill, a sum that wanders, or two memory instructions
    back to back in its main loop leave the matrix core idle. Checked on the generated code (compiled for the device only):
    no scratch; every MFMA adds into the accumulation registers it reads (or starts them from zero), 256 of them; in the
    main loop an MFMA sits between any two copies or fragment reads; the epilogue reads
    the sums behind the wait states written in the source."""
    import re
    import subprocess
    from yan_amd.jit import cpp_format, generate
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    from yan_amd.jit_kernels import bf16_gemm
    dtype = getattr(torch, dtype_name)
    _, keys, arg_defs = bf16_gemm.dense_kernel_plan(8192, 8192, 8192, dtype, 256, 0)
    assert (keys['BLOCK_M'], keys['BLOCK_N'], keys['NUM_STAGES']) == (256, 256, 2)
    src, asm = tmp_path / 'kernel.cu', tmp_path / 'kernel.s'
    src.write_text(generate(bf16_gemm.includes, arg_defs, cpp_format(bf16_gemm.template, keys)))
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-device-only', '-S', '-std=c++20', '-O3',
                           f'--offload-arch={get_offload_arch()}', '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
                           f'-I{get_jit_include_dir()}', str(src), '-o', str(asm)])
    text = asm.read_text()
    assert set(re.findall(r'\.private_segment_fixed_size:\s+(\d+)', text)) == {'0'} and 'scratch_' not in text, 'a kernel spills'
    name = 'dense_gemm_mfma_4w' if dtype == torch.bfloat16 else 'fp16_gemm_cute_4w'
    start = next(i for i, line in enumerate(text.split('\n')) if re.match(rf'^_ZN3yan\d*{name}\w*:', line))
    lines = [line.split(';')[0].strip() for line in text.split('\n')[start + 1:]]
    lines = lines[:lines.index('s_endpgm')]
    lines = [line for line in lines if line and not line.startswith(('.', '//'))]
    mfma = re.compile(r'^v_mfma_f32_16x16x32_(?:bf16|f16) (a\[\d+:\d+\]), v\[\d+:\d+\], v\[\d+:\d+\], (a\[\d+:\d+\]|0)$')
    assert not [line for line in lines if line.startswith('v_mfma') and not mfma.match(line)]
    sums = set()
    for line in lines:
        found = mfma.match(line)
        if found:
            assert found.group(2) in (found.group(1), '0'), line
            lo, hi = map(int, re.match(r'a\[(\d+):(\d+)\]', found.group(1)).groups())
            sums.update(range(lo, hi + 1))
    assert sums == set(range(256))
    # the main loop: from the second barrier (the first opens the first k-tile of the walk) to the last MFMA
    barriers = [i for i, line in enumerate(lines) if line == 's_barrier']
    last_mfma = max(i for i, line in enumerate(lines) if mfma.match(line))
    loop = [line for line in lines[barriers[1] + 1:last_mfma + 1] if not line.startswith('s_') and not line.endswith(':')]
    heavy = [i for i, line in enumerate(loop) if line.startswith(('buffer_load', 'ds_read'))]
    assert len(heavy) >= (16 + 32) + (8 + 16)              # a k-tile of the loop and the second k-half of the first one
    assert all(any(mfma.match(line) for line in loop[i + 1:j]) for i, j in zip(heavy, heavy[1:])), 'two copies or fragment reads with no MFMA between them'
    after = lines[last_mfma + 1:]
    first_read = next(i for i, line in enumerate(after) if line.startswith('v_accvgpr_read'))
    assert sum(1 for line in after[:first_read] if line == 's_nop 15') >= 2


@pytest.mark.parametrize('shape', [(4096, 7168, 7168), (64, 4096, 7168), (4096, 5120, 5120)])
def test_fp8_kernels_of_the_baseline_shapes_do_not_spill(tmp_path, shape):
    """The FP8 main loop keeps 128 running sums, the fragments of a row of atoms and the scales in registers and sits close
    to the 256-register limit; a spill puts scratch loads among its copies, and every wait for one of them waits for all
    copies in flight (measured: a variant that spilled 260 bytes ran 2.3 times slower). Checked on the generated code,
    compiled for the device only."""
    import re
    import subprocess
    from yan_amd.jit import cpp_format, generate
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    _, keys, arg_defs, _, code_template = gemm.fp8_kernel_plan(*shape, 256, True)
    src, asm = tmp_path / 'kernel.cu', tmp_path / 'kernel.s'
    src.write_text(generate(gemm.includes, arg_defs, cpp_format(code_template, keys)))
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-device-only', '-S', '-std=c++20', '-O3',
                           f'--offload-arch={get_offload_arch()}', '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
                           f'-I{get_jit_include_dir()}', str(src), '-o', str(asm)])
    text = asm.read_text()
    assert re.findall(r'\.private_segment_fixed_size:\s+(\d+)', text) == ['0'], 'the kernel spills'
    assert 'scratch_' not in text
    assert all(int(n) <= 256 for n in re.findall(r'\.vgpr_count:\s+(\d+)', text))
    assert text.count('16x16x128_f8f6f4') >= 4


def test_tuner_rebuilds_when_a_callers_dict_changes_between_calls(monkeypatch):
    """A caller that reuses one mutable keys dict (the loop of the reference's tests/test_jit.py) gets the kernel of the
    keys it passes, not of the keys it passed last time; only read-only plan keys take the same-object short cut."""
    from yan_amd.jit_kernels import tuner as tuner_mod
    built = []

    def fake_build(name, arg_defs, code):
        built.append(code)
        return object()
    monkeypatch.setattr(tuner_mod, 'build', fake_build)
    t = tuner_mod.JITTuner()
    kw = dict(name='k', space=(), includes=(), arg_defs=(('x', int),), template='int v = {V};', args=(1,))
    keys = {'V': 1}
    first = t.compile_and_tune(keys=keys, **kw)
    assert t.compile_and_tune(keys=keys, **kw) is first and len(built) == 1
    keys['V'] = 2
    second = t.compile_and_tune(keys=keys, **kw)
    assert second is not first and len(built) == 2 and 'int v = 2;' in built[1]
    frozen = tuner_mod.FrozenKeys({'V': 1})
    assert t.compile_and_tune(keys=frozen, **kw) is first and t.compile_and_tune(keys=frozen, **kw) is first
    with pytest.raises(TypeError):
        frozen['V'] = 3


def test_compare_tensors_verdicts(capsys):
    """yan/jit_kernels/utils.py:138-179: element-wise and similarity modes, shape mismatch, unknown mode."""
    from yan_amd.jit_kernels import compare_tensors
    x = torch.arange(12, dtype=torch.float32).view(3, 4)
    assert compare_tensors(x, x.clone()) is True and compare_tensors(x, x.clone(), mode='similarity', verbose=False) is True
    y = x.clone()
    y[1, 2] += 0.5
    capsys.readouterr()
    assert compare_tensors(y, x, verbose=False) is False
    said = capsys.readouterr().out
    assert 'FAILED' in said and 'Max diff: 0.500000' in said and '[1, 2]' in said and 'Actual tensor' not in said
    assert compare_tensors(y, x, atol=1.0) is True
    assert compare_tensors(y, x, mode='similarity', diff_tolerance=1e-2) is True
    assert compare_tensors(y, x, mode='similarity', diff_tolerance=1e-9) is False
    assert compare_tensors(torch.zeros(3), torch.zeros(3), mode='similarity') is True
    assert compare_tensors(x, x[:2]) is False and compare_tensors(x, x, mode='cosine') is False


def test_split_k_workspaces_are_kept_per_stream_and_per_capture():
    """Bookkeeping of the Python entries' split-K workspaces: eager launches share a workspace per (device, stream), at
    most `max_eager` are kept; every capture gets its own, never shared with eager launches or another capture and never
    dropped; a workspace whose launch failed is cleared before its next use."""
    from yan_amd.jit_kernels.split_k import WorkspaceBook
    made, cleared = [], []
    book = WorkspaceBook(make=lambda: made.append(object()) or made[-1], clear=cleared.append, max_eager=3)
    w0 = book.get(0, 111)
    assert book.get(0, 111) is w0 and len(made) == 1
    w1 = book.get(0, 222)
    w2 = book.get(1, 111)
    assert len({id(w) for w in (w0, w1, w2)}) == 3
    # captures: keyed by the capture's id, not by the stream that records it
    c7 = book.get(0, 111, capture=7)
    assert c7 is not w0 and book.get(0, 111, capture=7) is c7 and book.get(0, 999, capture=7) is c7
    c8 = book.get(0, 111, capture=8)
    assert c8 is not c7 and book.get(1, 111, capture=7) is not c7
    assert len(made) == 6 and not cleared
    # a failed launch: cleared once, at the next use
    book.launch_failed(0, 222)
    assert not cleared
    assert book.get(0, 222) is w1 and cleared == [w1]
    assert book.get(0, 222) is w1 and cleared == [w1]
    book.launch_failed(0, 111, capture=7)           # the graph's own first node zeroes a capture's workspace
    assert book.get(0, 111, capture=7) is c7 and cleared == [w1]
    # eviction: the oldest eager workspace goes, captures stay
    book.launch_failed(0, 111)
    w3 = book.get(2, 5)
    assert (0, 111) not in book.eager and len(book.eager) == 3 and (0, 111) not in book.suspect
    assert book.get(0, 111) is not w0 and cleared == [w1]       # a fresh one: nothing to clear
    assert len(book.captures) == 3 and book.get(0, 1, capture=8) is c8 and w3 is book.get(2, 5)


def test_the_bf16_activation_entry_chains_the_quantiser_in_front_of_whatever_the_gemm_entry_runs():
    """`fp8_cast_chain_plan`: the keys of the GEMM plan the FP8 entry uses for the sizes (split-K plan, weight-streaming kernel
    or tiles) plus the scratch offset, a `launch` whose arguments are the GEMM's without the quantised operands, and code
    that calls the quantiser before the GEMM's launch; None when the codes do not fit the scratch."""
    import harness as testing
    from yan_amd.jit import cpp_format
    from yan_amd.jit_kernels.split_k import SPLIT_K_WORKSPACE_BYTES, WORKSPACE_ALLOCATION_BYTES
    assert WORKSPACE_ALLOCATION_BYTES == SPLIT_K_WORKSPACE_BYTES + gemm.CAST_SCRATCH_BYTES
    for m, n, k in testing.CAST_CHAIN_SHAPES:
        plan = gemm.fp8_cast_chain_plan(m, n, k, 256)
        if m * k + m * (k // 128) * 4 + 256 > gemm.CAST_SCRATCH_BYTES:
            assert plan is None
            continue
        name, keys, arg_defs, code_template, smem_size = plan
        split = gemm.fp8_split_k_plan(m, n, k, 256, True)
        inner_keys, inner_defs = (split[1], split[2]) if split is not None else gemm.fp8_kernel_plan(m, n, k, 256, True)[1:3]
        assert name == 'gemm_bf16_fp8_bf16_nt' and dict(keys) == {**inner_keys, 'SCRATCH_OFFSET': SPLIT_K_WORKSPACE_BYTES}
        assert [d[0] for d in arg_defs] == ['x', 'buffer', 'scratch_bytes'] + [d[0] for d in inner_defs if d[0] not in ('lhs', 'lhs_scales')]
        code = cpp_format(code_template, keys)
        assert code.index('launch_per_token_cast(') < code.index('__return_code = static_cast<int>(', code.index('launch_per_token_cast(') + 1)
        assert '{' + 'SCRATCH_OFFSET' + '}' not in code and smem_size > 0
    # without split-K (YAN_SPLIT_K=0 leaves the entries without memory of their own) the entry makes two calls; the plan for it is not asked
    assert gemm.fp8_cast_chain_plan(64, 4096, 7168, 256, False)[1].get('SPLIT_K') is None


def test_contiguous_kernel_waits_for_its_copies_between_two_tiles_of_a_walk(tmp_path):
    """Workgroups that walk several slots of `fp8_gemm_contiguous_rows_kernel` go from tall to flat tiles, whose LDS stages are laid out
    differently: every wave's copies have to land before the barrier between two slots. Checked on the generated code (the
    main loops wait for a count of their own): each barrier is found with the wait in front of it, and exactly one of
    them, the one that is followed by the jump back to the walk, waits for all copies."""
    import re
    import subprocess
    import harness as testing
    from yan_amd.jit import cpp_format, generate
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    from yan_amd.jit_kernels import m_grouped_gemm
    _, keys, arg_defs, template = testing.grouped_rows_on_device_plan(4, 4096, 7168)
    src, asm = tmp_path / 'kernel.cu', tmp_path / 'kernel.s'
    src.write_text(generate(m_grouped_gemm.includes, arg_defs, cpp_format(template, keys)))
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-device-only', '-S', '-std=c++20', '-O3',
                           f'--offload-arch={get_offload_arch()}', '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
                           f'-I{get_jit_include_dir()}', str(src), '-o', str(asm)])
    lines = [line.split(';')[0].strip() for line in asm.read_text().split('\n')]
    lines = [line for line in lines if line and not line.startswith('.') or line.endswith(':')]
    waits = [re.search(r'vmcnt\((\d+)\)', ' '.join(ln for ln in lines[i - 2:i] if ln.startswith('s_waitcnt')))
             for i, line in enumerate(lines) if line == 's_barrier']
    assert len(waits) >= 6 and sum(w is not None and int(w.group(1)) == 0 for w in waits) == 1


def test_streams_forked_inside_a_capture_get_a_workspace_each(monkeypatch):
    """Two streams that record into one capture are branches of the graph that may run side by side: their split-K launches must
    not meet in one workspace. Launches on one of them share theirs, and another capture gets others."""
    from yan_amd.jit_kernels import split_k
    made = []
    monkeypatch.setattr(split_k, '_book', split_k.WorkspaceBook(make=lambda: made.append(object()) or made[-1], clear=lambda w: None))
    monkeypatch.setattr(split_k, '_last', (None, None))
    monkeypatch.setattr(split_k, '_is_capturing', lambda: True)
    capture = [7]
    monkeypatch.setattr(split_k, 'capture_id', lambda stream: capture[0])
    monkeypatch.delenv('YAN_SPLIT_K', raising=False)
    device = torch.device('cuda', 0)
    main, token = split_k.split_k_workspace(device, 111)
    side, _ = split_k.split_k_workspace(device, 222)
    assert side is not main and split_k.split_k_workspace(device, 111)[0] is main and split_k.split_k_workspace(device, 222)[0] is side
    split_k.split_k_launch_failed(token)
    assert split_k.split_k_workspace(device, 111)[0] is main
    capture[0] = 8
    assert split_k.split_k_workspace(device, 111)[0] not in (main, side) and len(made) == 3


def test_a_thread_on_another_stream_cannot_slip_in_its_workspace(monkeypatch):
    """The latest eager workspace is remembered for the next call; a call that finds its own stream remembered must return that
    stream's workspace also when a thread on another stream is served between the look and the return."""
    from yan_amd.jit_kernels import split_k
    monkeypatch.setattr(split_k, '_book', split_k.WorkspaceBook(make=object, clear=lambda w: None))
    monkeypatch.setattr(split_k, '_last', (None, None))
    monkeypatch.setattr(split_k, '_is_capturing', lambda: False)
    monkeypatch.delenv('YAN_SPLIT_K', raising=False)
    device = torch.device('cuda', 0)
    mine, _ = split_k.split_k_workspace(device, 111)
    others = []

    class Stream(int):          # compared while the other thread gets its turn
        __hash__ = int.__hash__

        def __eq__(self, other):
            if not others:
                others.append(None)
                others[0] = split_k.split_k_workspace(device, 222)[0]
            return int(self) == int(other)

    assert split_k.split_k_workspace(device, Stream(111))[0] is mine
    assert others[0] is not None and others[0] is not mine


def test_contiguous_keys_may_name_any_tile_of_256_rows(tmp_path):
    """`Gemm<..., 256, BLOCK_N, ..., kNumStages, ..., GroupedContiguous>::run_grouped` takes every width and depth the tiles support,
    not only those a plan names: the static checks of host and device code pass for all of them."""
    import subprocess
    import harness as testing
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    src = tmp_path / 'keys.hip'
    calls = '\n'.join(f'    yan::Gemm<520, 384, 256, {n}, 128, 4, {stages}, 1, yan::GemmType::GroupedContiguous>::run_grouped('
                      'out, q, s, 1, 1, 0, q, s, g, 4, 256, 520, 384, nullptr, 0, 0);' for n, stages in testing.GROUPED_256_ROW_KEYS)
    src.write_text('#include "gemm/fp8_gemm.hpp"\nvoid keys(__hip_bfloat16* out, const void* q, const float* s, const int* g) {\n' + calls + '\n}\n')
    subprocess.check_call([get_hipcc_compiler()[0], '--cuda-device-only', '-fsyntax-only', '-std=c++20', f'--offload-arch={get_offload_arch()}',
                           f'-I{get_jit_include_dir()}', str(src)])


# (groups, rows, n, k): microseconds of the 128-row tile the cost table takes and of the kernel whose tiles follow the groups (MI355X,
# router-like layouts)
SHORT_GROUPS = {(49, 9856, 1344, 1280): (34.1, 40.1), (43, 7040, 2112, 1152): (32.7, 38.8), (46, 8320, 1344, 1024): (28.0, 31.9),
                (29, 3712, 4352, 2560): (67.8, 73.6), (33, 4608, 3392, 1792): (48.2, 51.8), (41, 8448, 1600, 1664): (40.3, 46.4),
                (21, 2688, 5824, 1536): (45.5, 46.9),
                (64, 8320, 7168, 2048): (190.5, 174.8), (32, 6144, 4096, 4096): (142.3, 130.0), (24, 3968, 2880, 2048): (46.2, 41.2),
                (23, 2944, 4032, 1664): (41.5, 38.9), (50, 9728, 1152, 1408): (36.0, 32.6), (10, 1280, 7168, 2048): (44.0, 33.9),
                (29, 6784, 4160, 1152): (66.7, 57.7), (13, 1920, 4992, 2560): (55.9, 42.0), (59, 11392, 6144, 2176): (223.7, 203.2)}


def test_short_contiguous_groups_get_the_kernel_that_measured_faster():
    for (groups, m, n, k), (fixed, follows) in SHORT_GROUPS.items():
        assert heuristics.get_contiguous_rows_on_device(m, n, k, 256, groups) == (follows < fixed), (groups, m, n, k)


def test_time_of_tall_and_flat_tiles_is_that_of_a_list_schedule():
    import heapq
    flat_time = heuristics._FP8_TILES[(128, 256)] / 2
    for cus in (1, 8, 80, 256):
        for tall in (0, 1, cus - 1, cus, cus + 3, 3 * cus + cus // 2):
            for flat in (0, 1, cus // 2, cus, 2 * cus + 5, 7 * cus):
                free = [0.0] * cus
                for time in [1.0] * tall + [flat_time] * flat:
                    heapq.heapreplace(free, free[0] + time)
                assert heuristics._tall_then_flat(tall, flat, cus) == pytest.approx(max(free)), (tall, flat, cus)


def test_long_contiguous_groups_get_256_by_128_tiles_where_these_are_more_than_a_round():
    for groups, m, n, k, tile in ((4, 11008, 1284, 256, (256, 128)), (10, 11136, 1408, 1280, (256, 128)), (10, 15104, 2112, 5760, (256, 128)), (6, 11264, 1408, 5504, (256, 128)),
                                  (4, 5504, 2944, 6528, (256, 128)), (6, 6784, 1152, 6912, (128, 128)), (4, 4352, 1856, 6912, (128, 128)),
                                  (11, 11136, 1408, 1280, (128, 128))):
        assert heuristics.get_best_grouped_fp8_config(m, n, k, 256, 1, 128, groups) == tile


@pytest.mark.parametrize('m,n,k', [(330, 3648, 256), (300, 4004, 256)])
def test_fp8_kernels_of_two_k_tiles_compile(tmp_path, m, n, k):
    """64 x 128 tiles with K = 256: every LDS address of the unrolled loop is known at compile time."""
    import subprocess
    from yan_amd.jit import cpp_format, generate
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    from yan_amd.jit_kernels import gemm
    _, keys, arg_defs, _, template = gemm.fp8_kernel_plan(m, n, k, 256, True)
    assert (keys['BLOCK_M'], keys['BLOCK_N']) == (64, 128)
    src = tmp_path / 'kernel.cu'
    src.write_text(generate(gemm.includes, arg_defs, cpp_format(template, keys)))
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-device-only', '-S', '-std=c++20', '-O3', f'--offload-arch={get_offload_arch()}',
                           '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', f'-I{get_jit_include_dir()}', str(src),
                           '-o', str(tmp_path / 'kernel.s')])


@pytest.mark.parametrize('tile,k', [((128, 128), 1152), ((128, 256), 768), ((256, 128), 512), ((256, 256), 384), ((256, 256), 1664)])
def test_fp8_tiles_do_not_spill_where_k_is_short(tmp_path, tile, k):
    import re
    import subprocess
    import harness as testing
    from yan_amd.jit import cpp_format, generate
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    from yan_amd.jit_kernels import gemm
    _, keys, arg_defs, template = testing.fp8_explicit_tile_plan(*tile, 4096, k)
    src, asm = tmp_path / 'kernel.cu', tmp_path / 'kernel.s'
    src.write_text(generate(gemm.includes, arg_defs, cpp_format(template, keys)))
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-device-only', '-S', '-std=c++20', '-O3', f'--offload-arch={get_offload_arch()}',
                           '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', f'-I{get_jit_include_dir()}', str(src), '-o', str(asm)])
    assert set(re.findall(r'vgpr_spill_count: *(\d+)', asm.read_text())) == {'0'}


def test_fp32_split_k_counts_the_rounds_of_the_fullest_xcd():
    """The parts of a tile run on one XCD: plans whose tiles divide badly over the eight of them measured 18 to 45 % slower than the
    unsplit kernel or another plan (640 x 320 x 7168 in five parts 49 us, unsplit 38; 128 x 2112 x 9001 on 128 x 64 tiles in seven
    82, on 64 x 64 56)."""
    from yan_amd.jit_kernels.utils import ceil_div
    assert heuristics.get_split_k_float_config(640, 320, 7168, 256) is None
    assert heuristics.get_split_k_float_config(640, 1088, 4099, 256) is None
    assert heuristics.get_split_k_float_config(1024, 576, 2149, 256) is None
    assert heuristics.get_split_k_float_config(128, 2112, 9001, 256) == (64, 64, 7)
    assert heuristics.get_split_k_float_config(128, 2112, 7168, 256) == (64, 64, 7)
    assert heuristics.get_split_k_float_config(128, 256, 8192, 256) == (32, 32, 8)
    # what is split ends sooner than it would unsplit by rounds and k-rows alone
    us = heuristics._FLOAT_US_PER_1024_K
    for m in (128, 384, 640, 1024):
        for n in range(64, 4097, 192):
            for k in (1100, 2050, 4099, 8192):
                plan = heuristics.get_split_k_float_config(m, n, k, 256)
                if plan is not None:
                    tile, split = plan[:2], plan[2]
                    rounds = ceil_div(ceil_div(ceil_div(m, tile[0]) * ceil_div(n, tile[1]), 8) * split, 32)
                    whole = heuristics.get_best_float_config(m, n, 256)
                    assert rounds * us[tile] / split < ceil_div(ceil_div(m, whole[0]) * ceil_div(n, whole[1]), 256) * us[whole]


def test_fp32_plans_on_the_bf16_cores_fit_their_workspace():
    from yan_amd.jit_kernels import simple_gemm, split_k
    from yan_amd.jit_kernels.utils import ceil_div
    assert heuristics.get_float_bf16x3_config(1024, 1024, 1023, 256) is None and heuristics.get_float_bf16x3_config(128, 2112, 7168, 256) == (128, 64, 7)
    for m in (128, 384, 1024, 4096):
        for n in range(64, 8193, 832):
            for k in (1, 300, 2050, 8191):
                plan = heuristics.get_float_bf16x3_config(m, n, k, 256)
                whole = heuristics.get_float_bf16x3_config(m, n, k, 256, may_split=False)
                assert (plan is None) == (whole is None) == (m * n * k < heuristics.FLOAT_BF16X3_MIN_MNK)
                if plan is not None:
                    tiles = ceil_div(m, plan[0]) * ceil_div(n, plan[1])
                    assert whole[2] == 1
                    assert plan[2] == 1 or (split_k.SPLIT_K_COUNTER_BYTES + tiles * plan[0] * plan[1] * plan[2] * 4 <= split_k.SPLIT_K_WORKSPACE_BYTES
                                            and tiles * 8 * 4 <= split_k.SPLIT_K_COUNTER_BYTES)
                    assert simple_gemm.float_bf16x3_plan(m, n, k, 256)[2] is (simple_gemm.split_k_arg_defs if plan[2] > 1 else simple_gemm.arg_defs)


def test_fp32_plans_on_the_bf16_cores_cut_k_as_the_fp32_cores_would():
    """The rounding of a sum grows with what is added up in a row: K is cut (by waves that share it, by parts) no less often than by the plan on the
    fp32 cores."""
    waves = {(256, 256): 1, (256, 128): 2, (128, 256): 2, (128, 128): 4, (128, 64): 4}
    checked = 0
    for m in range(128, 4097, 384):
        for n in range(256, 8193, 448):
            for k in (257, 300, 690, 1255, 3543, 8191):
                for may_split in (True, False):
                    plan = heuristics.get_float_bf16x3_config(m, n, k, 256, may_split)
                    if plan is None:
                        continue
                    on_fp32 = (may_split and heuristics.get_split_k_float_config(m, n, k, 256)) or (*heuristics.get_best_float_config(m, n, 256), 1)
                    assert waves[plan[:2]] * plan[2] >= (4 if on_fp32[0] < 128 else 1) * on_fp32[2], (m, n, k, plan, on_fp32)
                    checked += 1
    assert checked > 1500


@pytest.mark.parametrize('kind,streams_codes', [('per_token', False), ('per_block', True)])
def test_codes_of_activations_are_stored_for_the_gemm_behind(tmp_path, kind, streams_codes):
    """The GEMM that follows a per-token cast reads its codes from the caches: no store of them carries the non-temporal hint.
    Weights are quantised ahead of time, those of a large matrix go past the caches."""
    import re
    import subprocess
    from yan_amd.jit import cpp_format, generate
    from yan_amd.jit.compiler import get_hipcc_compiler, get_jit_include_dir, get_offload_arch
    from yan_amd.jit_kernels import fp8_cast
    _, keys, arg_defs, template = fp8_cast.cast_kernel_plan(kind, torch.bfloat16)
    src, asm = tmp_path / 'kernel.cu', tmp_path / 'kernel.s'
    src.write_text(generate(fp8_cast.includes, arg_defs, cpp_format(template, keys)))
    subprocess.check_call([get_hipcc_compiler()[0], '-x', 'hip', '--cuda-device-only', '-S', '-std=c++20', '-O3', f'--offload-arch={get_offload_arch()}',
                           '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', f'-I{get_jit_include_dir()}', str(src), '-o', str(asm)])
    text = asm.read_text()
    assert re.search(r'global_load\S* .* nt\b', text)
    assert bool(re.search(r'global_store\S* .* nt\b', text)) == streams_codes
