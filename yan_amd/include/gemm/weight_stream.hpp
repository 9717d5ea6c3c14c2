// GEMM for few activation rows, bound by streaming the weights out of HBM once: one workgroup per 8 to 64 weight rows, K shared
// out over its 8 waves, no meeting of workgroups. FP8 with 128-block scales (fp8_gemm_skinny.hpp) and bf16 / fp16
// (bf16_gemm_skinny.hpp) are launched from here; contracts as in fp8_gemm.hpp and bf16_gemm.hpp.
//   * Wave w owns the 128-byte K blocks w, w + 8, w + 16, ... and copies the tile's weight rows and all activation rows of up to 4 of
//     them ahead into LDS slots of its own (buffer_load .. lds): nothing is shared before the partial sums meet, so the main loop
//     has no barrier, only the wave's own counts of copies in flight.
//   * Whole 128-byte lines are what a compute unit copies fast. Read straight into fragments (16 rows at 16 or 64 bytes per lane
//     group) operands that sit in L2 come in at 40 bytes/ns per compute unit, 8 rows x 128 bytes at a time at 125 - 190, into registers or
//     into LDS alike. The kernel that loaded fragments, 1 row, FP8, weights cycling: 2112 x 7168 9.7 us, this one 5.3 (split K over 3
//     workgroups per tile, their sums meeting in memory: 8.5); 1024 x 7168 9.3 / 4.5 (7.5); bf16 4096 x 2048 6.9 / 4.9,
//     16 rows x 1984 x 4608 12.6 / 6.8 (split: 9.8).
//   * What bounds it: weights at 6 - 7 TB/s where every compute unit has a tile, else the tile's rows + activation rows, pulled at
//     about 62 bytes/ns per compute unit (half of them behind loads that go to HBM), + 3.3 us of launch, first loads and the sum.
//   * Every workgroup reads all activations; each starts at another K block and wraps around, which spreads the requests over them.
#pragma once

#include <hip/hip_runtime.h>

#include "utils.hpp"
#include "mfma_utils.hpp"
#include "tile_io.hpp"
#include "fp8_cast.hpp"

namespace yan {

// ROWS weight rows and A_ROWS activation rows per workgroup; a slot holds one K block of both and, with SCALES, a float per row.
// OPERANDS: kDense (16-bit), kScaled (FP8 with scales), or kCast, FP8 weights with bf16 activations: a wave quantises the K blocks it owns
// of all of them first, while its first weights are on the way (up to kCastSteps times 4 groups of 128 numbers, 1 KB of LDS each).
// Every workgroup repeats that, bound by vector arithmetic of about 0.3 us a step, where a launch of the quantiser costs 2.5 to 3 us:
// 1 x 2112 x 7168 7.9 -> 6.0 us call to call, 4 x 5120 x 8192 11.6 -> 10.9. Quantising a block right in front of its MFMA instead put 0.4 us
// per block into the waves' chain (2112 x 7168 8.0).
enum StreamOperands { kDense, kScaled, kCast };
constexpr int kCastSteps = 8;
// Activation rows a workgroup of kCast works with for m rows and that many K blocks, or 0 when a wave's share does not fit.
__host__ __device__ constexpr int cast_rows(int m, int num_k_blocks) {
    const int rows = m <= 1 ? 1 : m <= 2 ? 2 : m <= 4 ? 4 : 8;
    return m >= 1 && m <= 8 && ceil_div(num_k_blocks, 8) * rows <= 4 * kCastSteps ? rows : 0;
}
template <int ROWS, int A_ROWS, StreamOperands OPERANDS>
struct WeightStreamShape {
    static constexpr bool SCALES = OPERANDS != kDense, CAST = OPERANDS == kCast;
    static_assert(ROWS % 8 == 0 && (A_ROWS == 8 || A_ROWS % 16 == 0 || CAST) && A_ROWS <= (CAST ? 8 : kWaveSize));
    static constexpr int NUM_WAVES = 8;
    static constexpr int LOADS = ROWS / 8 + (CAST ? 0 : A_ROWS / 8 + (SCALES ? 1 : 0));
    static constexpr int SLOT  = ROWS * kRowBytes + (CAST ? 0 : A_ROWS * kRowBytes + (SCALES ? kWaveSize * 4 : 0));
    static constexpr int CODES = CAST ? kCastSteps * 1024 : 0;         // of a wave
    static constexpr int FIT   = (152 * 1024 / NUM_WAVES - CODES) / SLOT;
    static constexpr int DEPTH = FIT < 4 ? FIT : 4;         // 3 to 5 measure alike; 8 is slower on a row (more copies in front of the first sum)
    static constexpr int ATOMS = ceil_div(A_ROWS, 16), B_ATOMS = ceil_div(ROWS, 16);
    static constexpr bool TWO_SCALES = SCALES && 128 % ROWS != 0;       // a tile can lie in two blocks of 128 weight rows
    static_assert(DEPTH >= 1 && B_ATOMS * ATOMS <= NUM_WAVES && DEPTH * SLOT >= B_ATOMS * ATOMS * kWaveSize * 16 && (DEPTH - 1) * LOADS < kNoWaitVm);
};

// Wait for the oldest of a wave's blocks when `later` blocks of LOADS copies each were issued after it (at most MAX).
template <int LOADS, int MAX>
__device__ __forceinline__ void wait_for_block(int later) {
    if constexpr (MAX > 0) {
        if (later < MAX) return wait_for_block<LOADS, MAX - 1>(later);
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(MAX * LOADS, kNoWaitLgkm));
    asm volatile("" ::: "memory");
}

// SCALES: FP8 operands with a scale per row and K block of the activations and per 128 weight rows and K block; else 16-bit ones.
// SHAPE_N, SHAPE_K_BYTES: the sizes when known at compile time, or 0.
template <typename Atom, typename Out, int SHAPE_N, int SHAPE_K_BYTES, int ROWS, int A_ROWS, StreamOperands OPERANDS>
__global__ void __launch_bounds__(8 * kWaveSize)
weight_stream_kernel(const uint8_t* __restrict__ lhs, const float* __restrict__ lhs_scales, const uint8_t* __restrict__ rhs,
                     const float* __restrict__ rhs_scales, Out* __restrict__ out, int m, int n_rt, int k_bytes_rt, int sa_stride_m, int sa_stride_k) {
    using Shape = WeightStreamShape<ROWS, A_ROWS, OPERANDS>;
    constexpr bool SCALES = Shape::SCALES, CAST = Shape::CAST;
    constexpr int NUM_WAVES = Shape::NUM_WAVES, DEPTH = Shape::DEPTH, SLOT = Shape::SLOT, ATOMS = Shape::ATOMS, B_ATOMS = Shape::B_ATOMS;
    constexpr int A_AT = ROWS * kRowBytes, SCALES_AT = (ROWS + A_ROWS) * kRowBytes;         // within a slot
    const int n = SHAPE_N ? SHAPE_N : n_rt, k_bytes = SHAPE_K_BYTES ? SHAPE_K_BYTES : k_bytes_rt;
    const int num_k_blocks = k_bytes / kRowBytes;

    __shared__ __attribute__((aligned(1024))) uint8_t slots[NUM_WAVES * (DEPTH * SLOT + Shape::CODES)];

    const int n0 = blockIdx.x * ROWS;
    const int lane = get_lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int g = lane / 16, col = lane % 16, sub = lane / 8;

    const int a_pitch = CAST ? 2 * k_bytes : k_bytes;
    const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(lhs, uint32_t(m) * a_pitch);
    const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(rhs, uint32_t(n) * k_bytes);
    __amdgpu_buffer_rsrc_t rsrc_sa = rsrc_a;
    const float* sb_row = nullptr, *sb_next = nullptr;
    bool in_next[B_ATOMS];          // this lane's four sums of an atom are in the second block of 128 rows (it starts at a multiple of 8)
    if constexpr (SCALES) {
        if constexpr (!CAST) rsrc_sa = make_rsrc(lhs_scales, (uint32_t(m - 1) * sa_stride_m + uint32_t(num_k_blocks - 1) * sa_stride_k + 1) * 4);
        sb_row = rhs_scales + size_t(n0 / 128) * num_k_blocks;
        sb_next = rhs_scales + size_t(min(n0 / 128 + 1, ceil_div(n, 128) - 1)) * num_k_blocks;
#pragma unroll
        for (int i = 0; i < B_ATOMS; ++i) in_next[i] = n0 % 128 + i * 16 + 4 * g >= 128;
    }
    // A copy moves 8 rows of a block, swizzled as tile_io.hpp has it; rows past the end of either matrix read as zero.
    const uint32_t chunk = uint32_t((lane & 7) ^ sub) * kChunk;
    const uint32_t voff_b = uint32_t(n0 + sub) * k_bytes, voff_a = uint32_t(sub) * k_bytes;
    const uint32_t voff_sa = lane < m && lane < A_ROWS ? uint32_t(lane) * sa_stride_m * 4 : kOutOfRange;

    const int rot = (blockIdx.x * 7) % num_k_blocks;
    auto rotated = [&](int kb) { const int r = kb + rot; return r >= num_k_blocks ? r - num_k_blocks : r; };

    uint8_t* const own = slots + wave * (DEPTH * SLOT);
    [[maybe_unused]] uint8_t* const codes = slots + NUM_WAVES * (DEPTH * SLOT) + wave * Shape::CODES;
    auto issue = [&](int block, int slot) {
        const int kb = rotated(block);
        uint8_t* const to = own + slot * SLOT;
#pragma unroll
        for (int p = 0; p < ROWS / 8; ++p)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, YAN_LDS_PTR(to + p * 8 * kRowBytes), kChunk, voff_b + (chunk ^ (p & 1) * kChunk),
                                                     kb * kRowBytes + p * 8 * k_bytes, 0, 0);
        if constexpr (CAST) return;
#pragma unroll
        for (int p = 0; p < A_ROWS / 8; ++p)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, YAN_LDS_PTR(to + A_AT + p * 8 * kRowBytes), kChunk, voff_a + (chunk ^ (p & 1) * kChunk),
                                                     kb * kRowBytes + p * 8 * k_bytes, 0, 0);
        if constexpr (SCALES) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_sa, YAN_LDS_PTR(to + SCALES_AT), 4, voff_sa, kb * sa_stride_k * 4, 0, 0);
    };

    // Lane (col, g) holds chunks 2g and 2g + 1 of row `col` of an atom. Half an atom of 8 rows is read twice, its second sums go nowhere.
    auto offset = [&](int row, int c) { return row * kRowBytes + ((c ^ swizzle_of_row(row)) * kChunk); };
    const int row_a = A_ROWS < 16 ? col & (A_ROWS - 1) : col;
    const int b_lo = offset(col, 2 * g), b_hi = offset(col, 2 * g + 1), a_lo = A_AT + offset(row_a, 2 * g), a_hi = A_AT + offset(row_a, 2 * g + 1);
    const int half_lo = offset(col & 7, 2 * g), half_hi = offset(col & 7, 2 * g + 1);

    f32x4 acc[B_ATOMS][ATOMS];
#pragma unroll
    for (int i = 0; i < B_ATOMS; ++i)
#pragma unroll
        for (int j = 0; j < ATOMS; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // kCast: group q of a wave is row q % A_ROWS of its block q / A_ROWS; a step is four groups, 16 lanes and 256 bytes of bf16 each
    [[maybe_unused]] const int own_blocks = wave < num_k_blocks ? (num_k_blocks - 1 - wave) / NUM_WAVES + 1 : 0;
    [[maybe_unused]] const int steps = ceil_div(own_blocks * A_ROWS, 4);
    if constexpr (CAST) {
        for (int t = 0; t < steps; ++t) {
            const int q = 4 * t + g, row = q % A_ROWS, kb = rotated(min(wave + q / A_ROWS * NUM_WAVES, num_k_blocks - 1));
            const uint32_t from = row < m ? uint32_t(row) * a_pitch + uint32_t(kb) * (2 * kRowBytes) + col * kChunk : kOutOfRange;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, YAN_LDS_PTR(codes + t * 1024), kChunk, from, 0, 0, 0);
        }
    }
#pragma unroll
    for (int s = 0; s < DEPTH; ++s)
        if (wave + s * NUM_WAVES < num_k_blocks) issue(wave + s * NUM_WAVES, s);
    // The codes of a step and, behind them, its scales take the place of its bf16 numbers; arithmetic of per_token_cast_kernel.
    auto code_at = [&](int q, int c) { return q / 4 * 1024 + q % 4 * kRowBytes + ((c ^ (q % 4)) * kChunk); };
    auto scale_at = [&](int q) { return q / 4 * 1024 + 4 * kRowBytes + q % 4 * 4; };
    if constexpr (CAST) {
        wait_for_block<Shape::LOADS, DEPTH>(min(own_blocks, DEPTH));
#pragma unroll 2
        for (int t = 0; t < steps; ++t) {
            Raw8<__hip_bfloat16> x;
            x.w[0] = *reinterpret_cast<const i32x4*>(codes + t * 1024 + lane * kChunk);
            const F32x8 f = to_f32(x);
            const float amax = fmaxf(max_over_16_lanes(abs_max8(f)), 1e-4f);
            const uint2 packed = quantise8(f, kFp8Max / amax);
            *reinterpret_cast<uint2*>(codes + code_at(4 * t + g, col / 2) + col % 2 * 8) = packed;
            if (col == 0) *reinterpret_cast<float*>(codes + scale_at(4 * t + g)) = amax / kFp8Max;
        }
    }
    for (int first = wave; first < num_k_blocks; first += DEPTH * NUM_WAVES) {
#pragma unroll
        for (int s = 0; s < DEPTH; ++s) {
            const int block = first + s * NUM_WAVES;
            if (block >= num_k_blocks) break;
            float sb = 0.f, sb2 = 0.f;
            if constexpr (SCALES) sb = sb_row[rotated(block)];
            if constexpr (Shape::TWO_SCALES) sb2 = sb_next[rotated(block)];
            wait_for_block<Shape::LOADS, DEPTH - 1>((num_k_blocks - 1 - block) / NUM_WAVES);
            const uint8_t* const from = own + s * SLOT;
            i32x4 b[B_ATOMS][2], a[ATOMS][2];
            float scale[ATOMS];
#pragma unroll
            for (int i = 0; i < B_ATOMS; ++i) {
                const bool half = i * 16 + 8 == ROWS;
                b[i][0] = *reinterpret_cast<const i32x4*>(from + (half ? half_lo : b_lo) + i * 16 * kRowBytes);
                b[i][1] = *reinterpret_cast<const i32x4*>(from + (half ? half_hi : b_hi) + i * 16 * kRowBytes);
            }
#pragma unroll
            for (int j = 0; j < ATOMS; ++j) {
                if constexpr (CAST) {
                    const int q = (block / NUM_WAVES) * A_ROWS + row_a;
                    a[j][0] = *reinterpret_cast<const i32x4*>(codes + code_at(q, 2 * g));
                    a[j][1] = *reinterpret_cast<const i32x4*>(codes + code_at(q, 2 * g + 1));
                    scale[j] = *reinterpret_cast<const float*>(codes + scale_at(q));
                } else {
                    a[j][0] = *reinterpret_cast<const i32x4*>(from + a_lo + j * 16 * kRowBytes);
                    a[j][1] = *reinterpret_cast<const i32x4*>(from + a_hi + j * 16 * kRowBytes);
                    if constexpr (SCALES) scale[j] = *reinterpret_cast<const float*>(from + SCALES_AT + (j * 16 + col) * 4);
                }
            }
            // the slot is read: its next block may come
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(kNoWaitVm, 0));
            asm volatile("" ::: "memory");
            if (block + DEPTH * NUM_WAVES < num_k_blocks) issue(block + DEPTH * NUM_WAVES, s);
#pragma unroll
            for (int j = 0; j < ATOMS; ++j)
#pragma unroll
                for (int i = 0; i < B_ATOMS; ++i) {
                    if constexpr (SCALES) {
                        const i32x8 bf = {b[i][0][0], b[i][0][1], b[i][0][2], b[i][0][3], b[i][1][0], b[i][1][1], b[i][1][2], b[i][1][3]};
                        const i32x8 af = {a[j][0][0], a[j][0][1], a[j][0][2], a[j][0][3], a[j][1][0], a[j][1][1], a[j][1][2], a[j][1][3]};
                        const f32x4 p = Atom::mma(bf, af, f32x4{0.f, 0.f, 0.f, 0.f});
                        const float ab = scale[j] * (Shape::TWO_SCALES && in_next[i] ? sb2 : sb);
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(p[r], ab, acc[i][j][r]);
                    } else {
                        using Frag = typename Atom::Frag;
                        acc[i][j] = Atom::mma(__builtin_bit_cast(Frag, b[i][0]), __builtin_bit_cast(Frag, a[j][0]), acc[i][j]);
                        acc[i][j] = Atom::mma(__builtin_bit_cast(Frag, b[i][1]), __builtin_bit_cast(Frag, a[j][1]), acc[i][j]);
                    }
                }
        }
    }

    // The partial sums of the 8 waves meet in their slots (a wave has no copy in flight and no slot to read any more).
#pragma unroll
    for (int i = 0; i < B_ATOMS; ++i)
#pragma unroll
        for (int j = 0; j < ATOMS; ++j) *reinterpret_cast<f32x4*>(own + ((i * ATOMS + j) * kWaveSize + lane) * 16) = acc[i][j];
    __syncthreads();
    if (wave < B_ATOMS * ATOMS) {
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NUM_WAVES; ++w) sum += *reinterpret_cast<const f32x4*>(slots + w * (DEPTH * SLOT) + (wave * kWaveSize + lane) * 16);
        // the 4 registers are weight rows nn .. nn + 3 of activation row mm
        const int row = wave / ATOMS * 16 + 4 * g, nn = n0 + row, mm = wave % ATOMS * 16 + col;
        if (mm < m && row < ROWS && nn < n) *reinterpret_cast<decltype(pack4(sum, Out{}))*>(out + size_t(mm) * n + nn) = pack4(sum, Out{});
    }
}

// Launch for m <= 16 * TM. Workgroups take as few weight rows as fit the chip (or the cap of `num_sms` workgroups) in one round: less to
// pull for each of them, and more of them. 8 rows: 1472 x 15104, one row, FP8, 6.9 us (16 rows: 8.2); 16 where 8 take two rounds:
// 4096 x 7168 7.0 us (8: 7.4); 24 for 8 x 4100 x 16384 14.0 (32: 15.6); 32 for 32 x 7168 x 2048 in bf16 8.0 us (16, two rounds: 10.2). Beyond that
// up to 32 activation rows (one sum per wave): 40 for 32 x 8200 x 8192 15.3 (48: 16.3; 64: 19.8; tiles: 25.7), 48 for 32 x 12288 x 2048 7.3
// (64: 7.9; tiles: 10.0), then 64: with 56 HBM-bound shapes lose (13000 x 16384 bf16 70.5 -> 74.2). False when a 32-bit offset does not reach.
template <typename Atom, typename Out, int SHAPE_N, int SHAPE_K_BYTES, int TM, StreamOperands OPERANDS, int CAST_ROWS = 0>
inline bool launch_weight_stream(const void* lhs, const float* lhs_scales, int sa_stride_m, int sa_stride_k, const void* rhs, const float* rhs_scales,
                                 void* out, int m, int n, int k_bytes, int num_sms, hipStream_t stream) {
    if (uint64_t(16 * TM) * k_bytes * (OPERANDS == kCast ? 2 : 1) >= kOutOfRange) return false;
    const int cus = num_sms > 0 && num_sms < device_cu_count() ? num_sms : device_cu_count();
    auto launch = [&]<int ROWS, int A_ROWS>() {
        // the last workgroup's rows lie up to ROWS - 1 behind the matrix
        if ((uint64_t(n) + (ROWS < 16 ? 16 : ROWS)) * k_bytes >= kOutOfRange) return false;
        hipLaunchKernelGGL((weight_stream_kernel<Atom, Out, SHAPE_N, SHAPE_K_BYTES, ROWS, A_ROWS, OPERANDS>), dim3(ceil_div(n, ROWS)), dim3(8 * kWaveSize), 0,
                           stream, static_cast<const uint8_t*>(lhs), lhs_scales, static_cast<const uint8_t*>(rhs), rhs_scales,
                           static_cast<Out*>(out), m, n, k_bytes, sa_stride_m, sa_stride_k);
        return true;
    };
    auto rows = [&]<int A_ROWS>() {
        if (ceil_div(n, 8) <= cus) return launch.template operator()<8, A_ROWS>();
        if (ceil_div(n, 16) <= cus) return launch.template operator()<16, A_ROWS>();
        if (ceil_div(n, 24) <= cus) return launch.template operator()<24, A_ROWS>();
        if constexpr (TM <= 2) {
            if (ceil_div(n, 32) > cus) {
                if (ceil_div(n, 40) <= cus) return launch.template operator()<40, A_ROWS>();
                if (ceil_div(n, 48) <= cus) return launch.template operator()<48, A_ROWS>();
                return launch.template operator()<64, A_ROWS>();
            }
        }
        return launch.template operator()<32, A_ROWS>();
    };
    if constexpr (OPERANDS == kCast) return rows.template operator()<CAST_ROWS>();
    else if constexpr (TM == 1) return m <= 8 ? rows.template operator()<8>() : rows.template operator()<16>();
    else return rows.template operator()<16 * TM>();
}

} // namespace yan
