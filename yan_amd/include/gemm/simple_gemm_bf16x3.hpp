// C = alpha * A . B^T + beta * C in fp32 on the bf16 matrix cores of gfx950: operands, layouts and result of simple_gemm.hpp, every fp32
// number taken apart into three bf16 numbers that add up to it.
//
//   x = h + m + l,  h = bf16(x), m = bf16(x - h), l = x - h - m          (24 bits of mantissa are three times eight; exact)
//   a b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh) + what is below 2^-24 |a b|
//
// Six products on cores of sixteen times the rate. bf16 has the exponents of fp32, products of two bf16 numbers are exact, and sixteen
// of them are added up per rounding, where the fp32 instruction adds two: against 64 bits the result is the closer one (relative error,
// N(0, 1) operands, K = 256 / 1024 / 7168: 2.9e-7 / 5.8e-7 / 1.5e-6 on the fp32 cores, 2.4e-7 / 4.9e-7 / 1.35e-6 here before K is split;
// positive and widely spread operands likewise). Where a number does not come apart (below 2^-110 with bits beyond the third bf16) is
// noticed: the workgroup stops there and goes on, from that k-tile to its last, on the fp32 cores. Where the sums are not finite in the end
// (infinities, NaN, sums that left the range) it runs its tile again there, from zero: the results are those of simple_gemm.hpp then.
// 4096^2 x 2048 with such a number in every row's first k-tile: 487 us (465 on the fp32 cores alone; 800 when such a tile ran on both from
// end to end); 128 x 2112 x 7168 48 (43; 72); NaN in every tile 755 and 64. Looking for them k-tile by k-tile costs the others 0.8 %.
//
// * Macro tiles as there, staged as they lie (a k-row of a tile is contiguous); a lane reads VM neighbouring rows of eight k-rows, which
//   are the rows of its VM atoms, and takes them apart in registers: 12 vector instructions for two numbers. 8 waves with slabs of
//   128 x 64 (64 x 64 on the 128 x 64 tile); waves that share a slab take 16 k-rows of a k-tile each (K_SPLIT).
// * The two waves of a SIMD take turns: while one takes its k-tile apart (288 instructions on a 128 x 64 slab) the other has 48 MFMAs of 32
//   cycles. Both kinds of work mixed in every wave were slower: 128 x 128 tiles 0.97 us a k-tile of 32, 0.74 in turns.
// * What bounds it: with few workgroups 1.48 us for 16 k-rows of a 256 x 256 tile (1.28 are MFMAs at 2.4 GHz), with all 256 compute units at
//   work 2.1 to 2.5, the power limit. 8192 x 8192 x 4096 3650 -> 2280 us (241 TFLOP/s; the fp32 cores peak at 157), 4096^2 x 2048
//   522 -> 297, 2048 x 1664 x 7227 427 -> 235, 128 x 2112 x 7168 with beta = 0 45 -> 32. Small problems stay on the fp32 cores: a tile here costs 5 to 10 us
//   besides its k-tiles (get_float_bf16x3_config).
#pragma once

#include "simple_gemm.hpp"

namespace yan {

template <int V> using template_int = std::integral_constant<int, V>;

template <int BLOCK_M_, int BLOCK_N_, int WAVES_M_, int WAVES_N_, int K_SPLIT_, int STAGES_>
struct SplitFloatShape {
    static constexpr int BLOCK_M = BLOCK_M_, BLOCK_N = BLOCK_N_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, K_SPLIT = K_SPLIT_, STAGES = STAGES_;
    static constexpr int NUM_WAVES = WAVES_M * WAVES_N * K_SPLIT, BLOCK_K = 16 * K_SPLIT;      // a wave takes one 16-deep step of a k-tile
    static constexpr int WTM = BLOCK_M / WAVES_M, WTN = BLOCK_N / WAVES_N, VM = WTM / 32, VN = WTN / 32;
    static constexpr int A_BYTES = BLOCK_K * BLOCK_M * 4, B_BYTES = BLOCK_K * BLOCK_N * 4, STAGE_BYTES = A_BYTES + B_BYTES;
    static constexpr int A_COPIES = A_BYTES / 1024, B_COPIES = B_BYTES / 1024, OPS = (A_COPIES + B_COPIES) / NUM_WAVES;
    static_assert(NUM_WAVES == 8 && VN == 2 && (VM == 2 || VM == 4));
    static_assert(A_COPIES % NUM_WAVES == 0 && B_COPIES % NUM_WAVES == 0);
    static_assert(STAGES >= 2 && STAGES * STAGE_BYTES < 160 * 1024 && (STAGES - 1) * OPS <= 63);
    // partial sums of the waves that share K, all of them or half at a time
    static constexpr int ROUNDS = NUM_WAVES * VM * VN * 16 * 256 <= STAGES * STAGE_BYTES ? 1 : 2;
    static_assert(K_SPLIT == 1 || NUM_WAVES * VM * VN * 16 * 256 / ROUNDS <= STAGES * STAGE_BYTES);
};
template <int BLOCK_M, int BLOCK_N> struct SplitFloatTile;
template <> struct SplitFloatTile<256, 256> : SplitFloatShape<256, 256, 2, 4, 1, 4> {};
template <> struct SplitFloatTile<256, 128> : SplitFloatShape<256, 128, 2, 2, 2, 3> {};
template <> struct SplitFloatTile<128, 256> : SplitFloatShape<128, 256, 1, 4, 2, 3> {};
template <> struct SplitFloatTile<128, 128> : SplitFloatShape<128, 128, 1, 2, 4, 2> {};
template <> struct SplitFloatTile<128, 64>  : SplitFloatShape<128, 64, 2, 1, 4, 3> {};

// Two fp32 numbers (one row, neighbouring k) as three pairs of bf16. The last remainder of a number above 2^-110 has at most eight bits,
// so it is a bf16 as it stands: `rest` collects what its lower half holds otherwise. (v_dot2_f32_bf16 would take a half out of a pair and
// subtract it in one instruction, but holds up the matrix core: 58 cycles for an MFMA and three of them, 33 with these.)
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l, uint32_t& rest) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    auto pair = [](float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2)); };
    auto first = [](uint32_t p) { return __builtin_bit_cast(float, p << 16); };
    auto second = [](uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); };
    h = pair(x0, x1);
    const float r0 = x0 - first(h), r1 = x1 - second(h);
    m = pair(r0, r1);
    const uint32_t s0 = __builtin_bit_cast(uint32_t, r0 - first(m)), s1 = __builtin_bit_cast(uint32_t, r1 - second(m));
    l = __builtin_amdgcn_perm(s1, s0, 0x07060302u);
    rest |= s0 | s1;
}

template <int BLOCK_M, int BLOCK_N, int SPLIT_K>
__device__ __forceinline__ void
float_gemm_split_body(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                      int m, int n, int k, int ldA, int ldB, int ldC, float alpha, float beta,
                      [[maybe_unused]] float* __restrict__ partials, [[maybe_unused]] unsigned* __restrict__ counters) {
    using Cfg = SplitFloatTile<BLOCK_M, BLOCK_N>;
    constexpr int VM = Cfg::VM, VN = Cfg::VN, BLOCK_K = Cfg::BLOCK_K, OPS = Cfg::OPS, STAGES = Cfg::STAGES, K_SPLIT = Cfg::K_SPLIT;
    using VecM = typename FloatVec<VM>::type;
    using VecN = typename FloatVec<VN>::type;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

    const XcdTileScheduler<> sched(m, n, BLOCK_M, BLOCK_N);
    int split = 0, tile_slot = int(blockIdx.x);
    TileCoord tile;
    if constexpr (SPLIT_K > 1) {
        // the parts of all tiles in one row, part by part, cut into eight: an XCD's share of it is one or two parts of K
        const int tiles_n = ceil_div(n, BLOCK_N), tiles = tiles_n * ceil_div(m, BLOCK_M), per_xcd = ceil_div(tiles * SPLIT_K, kNumXCD);
        const int at = int(blockIdx.x) % kNumXCD * per_xcd + int(blockIdx.x) / kNumXCD;
        split = at / tiles;
        tile_slot = at - split * tiles;
        tile = {tile_slot / tiles_n, tile_slot % tiles_n, int(blockIdx.x) / kNumXCD < per_xcd && split < SPLIT_K};
    } else {
        tile = sched.tile_of(tile_slot);
    }
    if (!tile.valid) return;
    const int all_k_tiles = ceil_div(k, BLOCK_K), per = ceil_div(all_k_tiles, SPLIT_K);
    const int kt_lo = min(split * per, all_k_tiles), kt_hi = min(kt_lo + per, all_k_tiles);
    const int k_end = SPLIT_K > 1 ? min(k, kt_hi * BLOCK_K) : k;
    const int m0 = tile.m_idx * BLOCK_M, n0 = tile.n_idx * BLOCK_N;

    const int lane = get_lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int ks = wave % K_SPLIT, wn = wave / K_SPLIT % Cfg::WAVES_N, wm = wave / (K_SPLIT * Cfg::WAVES_N);

    const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(A, k_end > 0 ? (uint32_t(k_end - 1) * uint32_t(ldA) + uint32_t(m)) * 4u : 0u);
    const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(B, k_end > 0 ? (uint32_t(k_end - 1) * uint32_t(ldB) + uint32_t(n)) * 4u : 0u);
    constexpr int A_LANES = BLOCK_M / 4, B_LANES = BLOCK_N / 4;
    constexpr int A_ROWS = kWaveSize / A_LANES, B_ROWS = kWaveSize / B_LANES;
    // rows past m and n read as zero: what lies there (padding, another matrix) could be NaN and send the tile to the fp32 cores
    const int row_a = m0 + (lane % A_LANES) * 4, row_b = n0 + (lane % B_LANES) * 4;
    const uint32_t voff_a = row_a < m ? (uint32_t(lane / A_LANES) * uint32_t(ldA) + uint32_t(row_a)) * 4u : kOutOfRange;
    const uint32_t voff_b = row_b < n ? (uint32_t(lane / B_LANES) * uint32_t(ldB) + uint32_t(row_b)) * 4u : kOutOfRange;
    auto copy_op = [&](int d, int kt, uint8_t* stage) {
        const int q = d * Cfg::NUM_WAVES + wave;
        if (d < Cfg::A_COPIES / Cfg::NUM_WAVES) {
            const uint32_t k_row = uint32_t(kt * BLOCK_K + q * A_ROWS);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, YAN_LDS_PTR(stage + q * 1024), kChunk, voff_a, k_row * uint32_t(ldA) * 4u, 0, 0);
        } else {
            const int qb = q - Cfg::A_COPIES;
            const uint32_t k_row = uint32_t(kt * BLOCK_K + qb * B_ROWS);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, YAN_LDS_PTR(stage + Cfg::A_BYTES + qb * 1024), kChunk, voff_b, k_row * uint32_t(ldB) * 4u, 0, 0);
        }
    };

    f32x16 acc[VM][VN];
    const int h = lane / 32, i = lane % 32;
    // lane (h, i) takes k-rows 8 h .. 8 h + 7 of its wave's step; row VM i + t of the slab belongs to atom t, column VN i + u to atom u
    const int raw_a = (16 * ks + 8 * h) * (BLOCK_M * 4) + (wm * Cfg::WTM + VM * i) * 4;
    const int raw_b = Cfg::A_BYTES + (16 * ks + 8 * h) * (BLOCK_N * 4) + (wn * Cfg::WTN + VN * i) * 4;

    __shared__ __attribute__((aligned(1024))) uint8_t ring[STAGES * Cfg::STAGE_BYTES];
    __shared__ int first_whole;                // the k-tile of this part from which on the fp32 cores go on, -1 if they start over
    if (threadIdx.x == 0) first_whole = 0x7fffffff;
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(kNoWaitVm, 0));        // before the first barrier
    auto clear = [&] {
#pragma unroll
        for (int t = 0; t < VM; ++t)
#pragma unroll
            for (int u = 0; u < VN; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t][u][r] = 0.f;
    };
    auto copies = [&](int kt, int stage) {
#pragma unroll
        for (int d = 0; d < OPS; ++d) copy_op(d, kt, ring + stage * Cfg::STAGE_BYTES);
    };

    struct Parts { u32x4 p[3]; };               // an atom's eight numbers of a lane, taken apart
    Parts fa[VM], fb[VN];
    auto read_a = [&](const uint8_t* stage, int j) { return *reinterpret_cast<const VecM*>(stage + raw_a + j * (BLOCK_M * 4)); };
    auto read_b = [&](const uint8_t* stage, int j) { return *reinterpret_cast<const VecN*>(stage + raw_b + j * (BLOCK_N * 4)); };
    auto take_apart = [&](int p, float x0, float x1, Parts& to, uint32_t& rest) {
        uint32_t x, y, z;
        split_pair(x0, x1, x, y, z, rest);
        to.p[0][p] = x; to.p[1][p] = y; to.p[2][p] = z;
    };
    // the six products of atoms t .. t + T - 1 with u .. u + U - 1, an accumulator's one after the other as far apart as they go
    auto multiply = [&](const Parts (&a)[VM], const Parts (&b)[VN], auto t0, auto tn, auto u0, auto un) {
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};      // small terms first
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int t = decltype(t0)::value; t < decltype(tn)::value; ++t)
#pragma unroll
                for (int u = decltype(u0)::value; u < decltype(un)::value; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[t].p[PA[q]]), __builtin_bit_cast(bf16x8, b[u].p[PB[q]]),
                                                                        acc[t][u], 0, 0, 0);
    };
    auto meet = [&](auto outstanding) {
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(decltype(outstanding)::value, kNoWaitLgkm));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto next_stage = [](int st) { return st + 1 == STAGES ? 0 : st + 1; };
    auto prev_stage = [](int st) { return st == 0 ? STAGES - 1 : st - 1; };
    clear();
    const int k_tiles = kt_hi - kt_lo;
    int done = 0;                   // k-tiles taken apart, the same for all waves
    uint32_t missing = 0;           // bit i: the k-tile i before the last of them had a number in it, of this wave's, that does not come apart
    const template_int<0> c0;
    const template_int<1> c1;
    const template_int<2> c2;
    {
        // The two waves of a SIMD (w and w + 4) take turns: while one takes its operands apart the other multiplies. The second of them
        // multiplies, in every k-tile, what it took apart in the one before.
#pragma unroll
        for (int t = 0; t < STAGES - 1; ++t) copies(kt_lo + t, t);
        int st = 0;
        // True once all waves know of a k-tile that one of them could not take apart: the one before this. Its products are left to the fp32
        // cores, which take over from there.
        auto convert = [&]() -> bool {
            const uint8_t* stage = ring + st * Cfg::STAGE_BYTES;
            const int noticed = first_whole;        // (an atomic or volatile load has the compiler wait for every copy in front of it)
            uint32_t rest = 0;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const VecM x = read_a(stage, 2 * p), y = read_a(stage, 2 * p + 1);
                const VecN v = read_b(stage, 2 * p), w = read_b(stage, 2 * p + 1);
#pragma unroll
                for (int t = 0; t < VM; ++t) take_apart(p, x[t], y[t], fa[t], rest);
#pragma unroll
                for (int u = 0; u < VN; ++u) take_apart(p, v[u], w[u], fb[u], rest);
            }
            missing <<= 1;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64((rest & 0xffffu) != 0) != 0, 0)) {
                missing |= 1;
#pragma unroll
                for (int t = 0; t < VM; ++t)
#pragma unroll
                    for (int q = 0; q < 3; ++q) fa[t].p[q] = u32x4{0, 0, 0, 0};
                if (lane == 0) __hip_atomic_fetch_min(&first_whole, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __builtin_amdgcn_s_waitcnt(waitcnt_imm(kNoWaitVm, 0));        // before the next barrier
            }
            __builtin_amdgcn_sched_barrier(0);
            // what others note in this k-tile may or may not be in `noticed`, and is no reason yet
            ++done;
            return __builtin_amdgcn_readfirstlane(noticed) < done - 1 || done == k_tiles;
        };
        // the copies of k-tile kt go into the stage of the k-tile in front of this one, which everybody has read
        auto multiply_and_copy = [&](int kt) {
            uint8_t* const left = ring + prev_stage(st) * Cfg::STAGE_BYTES;
            multiply(fa, fb, c0, template_int<VM>{}, c0, c2);
#pragma unroll
            for (int d = 0; d < OPS; ++d) copy_op(d, kt, left);
#pragma unroll
            for (int d = 0; d < OPS; ++d) {
                __builtin_amdgcn_sched_group_barrier(0x008, 6 * VM * VN / OPS / 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        if (wave < 4) {
            for (bool enough = k_tiles == 0; __builtin_expect(!enough, 1);) {
                meet(template_int<(STAGES - 2) * OPS>{});
                enough = convert();
                multiply_and_copy(kt_lo + done + STAGES - 2);
                st = next_stage(st);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int t = 0; t < VM; ++t) fa[t].p[q] = u32x4{0, 0, 0, 0};
#pragma unroll
                for (int u = 0; u < VN; ++u) fb[u].p[q] = u32x4{0, 0, 0, 0};
            }
            for (bool enough = k_tiles == 0; __builtin_expect(!enough, 1);) {
                meet(template_int<(STAGES - 2) * OPS>{});
                multiply_and_copy(kt_lo + done + STAGES - 1);
                enough = convert();
                st = next_stage(st);
            }
            multiply(fa, fb, c0, template_int<VM>{}, c0, c2);
        }
    }
    // The fp32 matrix cores take the k-tiles from the first on that did not come apart (numbers below 2^-110); of the two before the waves
    // stopped, what is missing. Where the sums so far are not finite (infinities, NaN, sums that left the range) they take all, from zero.
    float inf[4] = {0.f, 0.f, 0.f, 0.f};                    // NaN once a sum is not finite
#pragma unroll
    for (int t = 0; t < VM; ++t)
#pragma unroll
        for (int u = 0; u < VN; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) inf[r % 4] = __builtin_fmaf(acc[t][u][r], 0.f, inf[r % 4]);
    if ((inf[0] + inf[1]) + (inf[2] + inf[3]) != 0.f) first_whole = -1;
    wait_for_copies();
    __syncthreads();
    int from = __builtin_amdgcn_readfirstlane(first_whole);
    if (from < 0) {
        clear();
        from = done = 0;
    }
    if (from < k_tiles) {
        int st = 0;
#pragma unroll
        for (int t = 0; t < STAGES - 1; ++t) copies(kt_lo + from + t, t);
        for (int s = from; s < k_tiles; ++s) {
            meet(template_int<(STAGES - 2) * OPS>{});
            copies(kt_lo + s + STAGES - 1, prev_stage(st));
            // lane group h takes k-row 2 kp + h
            const uint8_t* pa = ring + st * Cfg::STAGE_BYTES + (16 * ks + h) * (BLOCK_M * 4) + (wm * Cfg::WTM + VM * i) * 4;
            const uint8_t* pb = ring + st * Cfg::STAGE_BYTES + Cfg::A_BYTES + (16 * ks + h) * (BLOCK_N * 4) + (wn * Cfg::WTN + VN * i) * 4;
            if (s >= done || (missing >> (done - 1 - s) & 1)) {
                VecM a[2];
                VecN b[2];
                auto fetch = [&](int kp) {
                    a[kp & 1] = *reinterpret_cast<const VecM*>(pa + kp * (2 * BLOCK_M * 4));
                    b[kp & 1] = *reinterpret_cast<const VecN*>(pb + kp * (2 * BLOCK_N * 4));
                };
                fetch(0);
#pragma unroll
                for (int kp = 0; kp < 8; ++kp) {
                    if (kp < 7) fetch(kp + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = 0; t < VM; ++t)
#pragma unroll
                        for (int u = 0; u < VN; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[kp & 1][t], b[kp & 1][u], acc[t][u], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            st = next_stage(st);
        }
        wait_for_copies();
        __syncthreads();
    }

    constexpr int QUADS = 4 / K_SPLIT;
    const int first_quad = ks * QUADS;
    f32x4 sums[VM * VN * QUADS];
    auto sum_of = [&](int t, int u, int q) -> f32x4& { return sums[(t * VN + u) * QUADS + q]; };
    auto quad_of = [&](int t, int u, int q) { return f32x4{acc[t][u][4 * q], acc[t][u][4 * q + 1], acc[t][u][4 * q + 2], acc[t][u][4 * q + 3]}; };
    constexpr int QUAD_VECS = VM * VN * kWaveSize;
    [[maybe_unused]] f32x4* const vecs = reinterpret_cast<f32x4*>(ring);
    if constexpr (K_SPLIT == 4) {
        // wave ks finishes quad ks; with room for half of the sums the quads go through two at a time
        constexpr int PER_ROUND = 4 / Cfg::ROUNDS;
        f32x4* slab = vecs + (wave / 4) * (4 * PER_ROUND * QUAD_VECS);         // [part][quad][t, u][lane]
#pragma unroll
        for (int round = 0; round < Cfg::ROUNDS; ++round) {
            if (round) __syncthreads();
#pragma unroll
            for (int t = 0; t < VM; ++t)
#pragma unroll
                for (int u = 0; u < VN; ++u)
#pragma unroll
                    for (int q = 0; q < PER_ROUND; ++q)
                        slab[(ks * PER_ROUND + q) * QUAD_VECS + (t * VN + u) * kWaveSize + lane] = quad_of(t, u, round * PER_ROUND + q);
            __syncthreads();
            if (ks / PER_ROUND == round) {
#pragma unroll
                for (int t = 0; t < VM; ++t)
#pragma unroll
                    for (int u = 0; u < VN; ++u) {
                        const f32x4* mine = slab + ks % PER_ROUND * QUAD_VECS + (t * VN + u) * kWaveSize + lane;
                        constexpr int PART = PER_ROUND * QUAD_VECS;
                        sum_of(t, u, 0) = ((mine[0] + mine[PART]) + mine[2 * PART]) + mine[3 * PART];
                    }
            }
        }
    } else if constexpr (K_SPLIT == 2) {
        // the two waves swap halves: quads 0, 1 are finished by the first, 2, 3 by the second
        f32x4* mine = vecs + wave * (2 * QUAD_VECS), *other = vecs + (wave ^ 1) * (2 * QUAD_VECS);
        auto swap = [&](auto half) {
            constexpr int H = decltype(half)::value;
#pragma unroll
            for (int t = 0; t < VM; ++t)
#pragma unroll
                for (int u = 0; u < VN; ++u)
#pragma unroll
                    for (int q = 0; q < 2; ++q) mine[q * QUAD_VECS + (t * VN + u) * kWaveSize + lane] = quad_of(t, u, 2 * (1 - H) + q);
            __syncthreads();
#pragma unroll
            for (int t = 0; t < VM; ++t)
#pragma unroll
                for (int u = 0; u < VN; ++u)
#pragma unroll
                    for (int q = 0; q < 2; ++q) sum_of(t, u, q) = quad_of(t, u, 2 * H + q) + other[q * QUAD_VECS + (t * VN + u) * kWaveSize + lane];
        };
        if (ks == 0) swap(template_int<0>{});
        else swap(template_int<1>{});
    } else {
#pragma unroll
        for (int t = 0; t < VM; ++t)
#pragma unroll
            for (int u = 0; u < VN; ++u)
#pragma unroll
                for (int q = 0; q < QUADS; ++q) sum_of(t, u, q) = quad_of(t, u, q);
    }
    if constexpr (SPLIT_K > 1)
        if (!meet_partials<SPLIT_K, Cfg::NUM_WAVES, VM * VN * QUADS>([&](int v) -> f32x4& { return sums[v]; }, partials, counters,
                                                                     tile_slot, split, wave, lane)) return;

    // Epilogue: register r of quad q of an atom is MFMA row 8 q + 4 h + r, the lane MFMA column i.
    const int n_lane = n0 + wn * Cfg::WTN + VN * i;
    if (n_lane >= n) return;                                   // n % 4 == 0: a lane's two columns exist together
    auto row_of = [&](int q, int r, int t) { return m0 + wm * Cfg::WTM + VM * (8 * (first_quad + q) + 4 * h + r) + t; };
    auto store = [&](auto reads_c) {
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
            // what C holds, 4 * VM rows at a time, rows past m read the last one again (simple_gemm.hpp)
            VecN held[4][VM];
            if constexpr (decltype(reads_c)::value) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int t = 0; t < VM; ++t) held[r][t] = *reinterpret_cast<const VecN*>(C + size_t(min(row_of(q, r, t), m - 1)) * ldC + n_lane);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < VM; ++t) {
                    const int mm = row_of(q, r, t);
                    if (mm >= m) continue;
                    VecN v = {alpha * sum_of(t, 0, q)[r], alpha * sum_of(t, 1, q)[r]};
                    if constexpr (decltype(reads_c)::value) v += beta * held[r][t];
                    *reinterpret_cast<VecN*>(C + size_t(mm) * ldC + n_lane) = v;
                }
        }
    };
    if (beta != 0.f) store(std::true_type{});
    else store(std::false_type{});
}

template <int BLOCK_M, int BLOCK_N, int SPLIT_K>
__global__ void __launch_bounds__(8 * kWaveSize, 1)
gemm_cute_bf16x3(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                 int m, int n, int k, int ldA, int ldB, int ldC, float alpha, float beta,
                 float* __restrict__ partials, unsigned* __restrict__ counters) {
    float_gemm_split_body<BLOCK_M, BLOCK_N, SPLIT_K>(A, B, C, m, n, k, ldA, ldB, ldC, alpha, beta, partials, counters);
}

// With SPLIT_K > 1 `workspace` is that of the other split-K launchers (kSplitKCounterBytes of counters that are zero before and after
// every launch, then the partial sums); launches that share it must not overlap.
template <int BLOCK_M, int BLOCK_N, int SPLIT_K>
inline hipError_t launch_float_nt_bf16x3(int m, int n, int k, float alpha, const float* A, int ldA, const float* B, int ldB,
                                         float beta, float* C, int ldC, hipStream_t stream, void* workspace = nullptr, size_t workspace_bytes = 0) {
    if (m == 0 || n == 0) return hipSuccess;
    // (of the smallest tile: the k-rows fetched past the end, at most 256, stay far below the 1024 its check leaves room for)
    if (hipError_t e = check_float_args(m, n, k, A, ldA, B, ldB, C, ldC, 32, 32); e != hipSuccess) return e;
    uint32_t grid = uint32_t(XcdTileScheduler<>(m, n, BLOCK_M, BLOCK_N).grid_size());
    if constexpr (SPLIT_K > 1) {
        const uint64_t tiles = uint64_t(ceil_div(m, BLOCK_M)) * uint64_t(ceil_div(n, BLOCK_N));
        if (!workspace || tiles * SplitFloatTile<BLOCK_M, BLOCK_N>::NUM_WAVES * 4 > kSplitKCounterBytes) return hipErrorInvalidValue;
        if (kSplitKCounterBytes + tiles * SPLIT_K * BLOCK_M * BLOCK_N * 4 > workspace_bytes) return hipErrorInvalidValue;
        grid = uint32_t(ceil_div<uint64_t>(tiles * SPLIT_K, kNumXCD)) * kNumXCD;
    }
    hipLaunchKernelGGL((gemm_cute_bf16x3<BLOCK_M, BLOCK_N, SPLIT_K>), dim3(grid), dim3(8 * kWaveSize), 0, stream,
                       A, B, C, m, n, k, ldA, ldB, ldC, alpha, beta,
                       SPLIT_K > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kSplitKCounterBytes) : nullptr,
                       static_cast<unsigned*>(workspace));
    return hipGetLastError();
}

} // namespace yan
