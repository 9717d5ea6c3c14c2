// Quantisers that feed the block-scaled FP8 GEMM: fp32 / bf16 -> e4m3 codes + fp32 scales, in one pass over HBM.
//
//   per-token:  one scale per row and 128 consecutive K   (activations; lhs_scales of the GEMM)
//   per-block:  one scale per 128 x 128 block              (weights; rhs_scales of the GEMM)
//   amax = max |x| over the group, clamped from below at 1e-4;  q = e4m3(x * (448 / amax));  scale = amax / 448
//
// This is the step in front of the GEMM entry whose operand names the reference fixes
// (yan/jit_kernels/gemm.py:23-30: lhs, lhs_scales, rhs, rhs_scales); the reference itself has no quantiser. The
// arithmetic is the recipe callers of this convention type in torch, `(x.float() * (448 / amax)).to(float8_e4m3fn)`
// and `amax / 448`, with both quotients correctly rounded: fp32 IEEE divisions, one fp32 multiply, round-to-nearest-
// even conversion. (torch itself evaluates `448.0 / amax` as reciprocal(amax) * 448, an ulp away for some amax.)
//
// Both kernels are bound by HBM traffic: (2 or 4) bytes read + 1 byte written per element, plus 4 bytes per
// group. Sixteen lanes own one 128-element group at a time, 8 elements per lane, so a wave reads 1 KB (bf16) or
// 2 KB (fp32) of consecutive addresses per step and writes 512 B. At that traffic a wave has about 150 vector
// instructions per 1 KB of bf16 before arithmetic is the bound as well, so sources are held as they were loaded, maxima
// cross lanes on the DPP path, scales are divided and placed once per wave for all of its groups, and indices are 32 bits.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include "utils.hpp"

namespace yan {

constexpr float kFp8Max = 448.0f;

// How a launch treats the caches. Sources and codes that outgrow the L2s together (8 x 4 MB) only push each other out
// of them: past that size sources are moved with the non-temporal hint, and so are the codes of weights, which nobody reads
// for a while. Those of activations are read at once, by the GEMM behind, which finds them in the memory-side cache only if
// they were stored plainly: per-token cast and GEMM together, codes streamed / plain, 6144 x 7168 (x 2112 outputs) 117.5 / 114.9 us,
// 16384 x 7168 (x 2112) 293 / 276, 12288 x 4096 (x 512) 62.4 / 59.3. Small launches take the plain forms, which are as fast or
// faster (64 x 7168: 2.5 us plain, 2.7 with either hint). Measured cold and alone, bf16, token-contiguous scales, kPlain /
// kStreamSource / kStreamBoth: 4096 x 7168 (59 MB read, 29 written) 17.5 / 16.0 / 16.3 us, 16384 x 7168 64.0 / 61.7 / 59.3; per
// block 16384 x 7168 66.1 / 62.3 / 59.6.
enum CastStream { kPlain, kStreamSource, kStreamBoth };
constexpr long long kCastL2Bytes = 32ll << 20;
inline CastStream cast_stream(long long elements, int bytes_per_element, bool codes_read_next) {
    if (elements > kCastL2Bytes && !codes_read_next) return kStreamBoth;
    return elements * bytes_per_element > kCastL2Bytes ? kStreamSource : kPlain;
}

// Eight elements of a group as loaded, and as fp32: lane `part` of the group's sixteen has 8 part .. 8 part + 7 of bf16 and, so
// that every load instruction reads whole lines there too, 4 part .. 4 part + 3 and 64 further on of fp32 (two loads of
// neighbouring 16 bytes each read half of every line twice, which the non-temporal hint turns into traffic).
struct F32x8 { float v[8]; };
template <typename T> struct Raw8 { i32x4 w[sizeof(T) / 2]; };

template <bool STREAM, typename T>
__device__ __forceinline__ Raw8<T> load8(const T* group, int part) {
    const i32x4* from = reinterpret_cast<const i32x4*>(group) + part;
    Raw8<T> r;
#pragma unroll
    for (int i = 0; i < int(sizeof(T) / 2); ++i) r.w[i] = STREAM ? __builtin_nontemporal_load(from + 16 * i) : from[16 * i];
    return r;
}

template <typename T>
__device__ __forceinline__ F32x8 to_f32(const Raw8<T>& r) {
    static_assert(sizeof(T) == 2 || sizeof(T) == 4, "bf16 or fp32");
    F32x8 f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        uint32_t bits;
        if constexpr (sizeof(T) == 4) bits = uint32_t(r.w[i / 4][i % 4]);
        else bits = i % 2 ? uint32_t(r.w[0][i / 2]) & 0xffff0000u : uint32_t(r.w[0][i / 2]) << 16;
        f.v[i] = __builtin_bit_cast(float, bits);
    }
    return f;
}

__device__ __forceinline__ float abs_max8(const F32x8& x) {
    float a = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) a = fmaxf(a, fabsf(x.v[i]));
    return a;
}

// The codes of what load8 gave this lane, to the group's 128 bytes.
template <typename T, bool STREAM>
__device__ __forceinline__ void store_codes8(uint8_t* group, int part, uint2 codes) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const auto store = [](auto v, auto* to) {
        if constexpr (STREAM) __builtin_nontemporal_store(v, to);
        else *to = v;
    };
    if constexpr (sizeof(T) == 2) {
        store(u32x2{codes.x, codes.y}, reinterpret_cast<u32x2*>(group) + part);
    } else {
        store(codes.x, reinterpret_cast<uint32_t*>(group) + part);
        store(codes.y, reinterpret_cast<uint32_t*>(group) + 16 + part);
    }
}

// Eight e4m3 codes (OCP on gfx950, round to nearest even) of x * factor, packed little-endian in two dwords.
__device__ __forceinline__ uint2 quantise8(const F32x8& x, float factor) {
    int lo = 0, hi = 0;
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(x.v[0] * factor, x.v[1] * factor, lo, false);
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(x.v[2] * factor, x.v[3] * factor, lo, true);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(x.v[4] * factor, x.v[5] * factor, hi, false);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(x.v[6] * factor, x.v[7] * factor, hi, true);
    return make_uint2(uint32_t(lo), uint32_t(hi));
}

// Maximum over the 16 lanes that share a group (lanes 16g .. 16g+15 of the wave, a DPP row: four rotations of it). In
// floats, not in their bits: a lane whose last value is a signalling NaN holds a NaN, and that one must not win. Every lane
// of the wave has to be active.
template <int ROTATE>
__device__ __forceinline__ float rotate_in_16_lanes(float a) {
    constexpr int ROW_ROR = 0x120;
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, a), ROW_ROR + ROTATE, 0xf, 0xf, true));
}
__device__ __forceinline__ float max_over_16_lanes(float a) {
    a = fmaxf(a, rotate_in_16_lanes<8>(a));
    a = fmaxf(a, rotate_in_16_lanes<4>(a));
    a = fmaxf(a, rotate_in_16_lanes<2>(a));
    return fmaxf(a, rotate_in_16_lanes<1>(a));
}

// x [m, k] row-major with k % 128 == 0, m * k / 128 groups. Scale of (row, kb) goes to scales[row * stride_m + kb * stride_k].
// UNROLL groups per 16 lanes are in flight at once. A workgroup takes the 16 * UNROLL groups that follow each other in
// the order its scales are stored in: groups of one row and the next (row-major scales) or, BY_ROWS, the same K block of
// 16 * UNROLL rows (token-contiguous scales), so that its scales fill whole lines instead of 4 bytes in each of
// 32 lines. 4096 x 7168 bf16 with token-contiguous scales, cold: 20.6 us with a 64-bit division per group, shuffles and groups
// along the row, 19.1 without the first two, 17.5 by rows, 16.0 streaming the source; row-major scales 18.8 -> 15.6;
// 16384 x 7168 63.5 -> 58.6 and 60.4 -> 54.8, fp32 105 -> 96 and 103 -> 90; 64 x 7168, in front of a decode GEMM, 3.3 -> 2.5.
template <typename T, int UNROLL, bool BY_ROWS, CastStream STREAM>
__global__ void __launch_bounds__(256)
per_token_cast_kernel(const T* __restrict__ x, uint8_t* __restrict__ q, float* __restrict__ scales,
                      uint32_t m, uint32_t k_blocks, long long stride_m, long long stride_k) {
    static_assert(UNROLL <= 16, "lane u of a group's sixteen finishes the scale of group u");
    const uint32_t part = threadIdx.x & 15, sub = threadIdx.x >> 4;         // 256 threads = 16 groups per step
    const uint32_t num_groups = m * k_blocks;                               // fits: see launch_per_token_cast
    uint32_t first, kb = 0;                                                 // first row of the workgroup, or first group
    if constexpr (BY_ROWS) {
        const uint32_t rows = blockIdx.x / k_blocks;
        kb = blockIdx.x - rows * k_blocks;
        first = rows * (16 * UNROLL);
    } else {
        first = blockIdx.x * (16 * UNROLL);
    }
    const uint32_t end = BY_ROWS ? m : num_groups;
    Raw8<T> v[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
        const uint32_t at = first + u * 16 + sub, group = BY_ROWS ? at * k_blocks + kb : at;
        v[u] = Raw8<T>{};
        if (at < end) v[u] = load8<STREAM != kPlain>(x + size_t(group) * 128, part);
    }
    float amax_of_part = 0.f;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
        const uint32_t at = first + u * 16 + sub, group = BY_ROWS ? at * k_blocks + kb : at;
        const F32x8 f = to_f32(v[u]);
        const float amax = fmaxf(max_over_16_lanes(abs_max8(f)), 1e-4f);
        if (part == u) amax_of_part = amax;
        if (at < end) store_codes8<T, STREAM == kStreamBoth>(q + size_t(group) * 128, part, quantise8(f, kFp8Max / amax));
    }
    const uint32_t at = first + part * 16 + sub;
    if (part < UNROLL && at < end) {
        const uint32_t row = BY_ROWS ? at : at / k_blocks, block = BY_ROWS ? kb : at - row * k_blocks;
        scales[row * stride_m + block * stride_k] = amax_of_part / kFp8Max;
    }
}

// w [n, k] row-major with k % 128 == 0: one workgroup per 128 x 128 block; rows past n count as zeros and are not
// written. scales [ceil(n/128), k/128] row-major.
// Cold, with the sources held as loaded and moved past the caches: 7168 x 7168 bf16 33.2 -> 27.6 us (5.6 TB/s),
// 16384 x 7168 68.7 -> 59.8, fp32 49.3 -> 44.2 and 109.8 -> 97.7.
template <typename T, CastStream STREAM>
__global__ void __launch_bounds__(256)
per_block_cast_kernel(const T* __restrict__ w, uint8_t* __restrict__ q, float* __restrict__ scales, int n, int k) {
    __shared__ float wave_max[4];
    const int k_blocks = k / 128;
    const int kb = blockIdx.x % k_blocks, nb = blockIdx.x / k_blocks;
    const int part = threadIdx.x & 15, row_in_step = threadIdx.x >> 4;      // 16 rows per step, 8 steps
    Raw8<T> v[8];       // as loaded: for bf16 half the registers of its fp32 values, twice the workgroups in flight
    float amax = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int row = nb * 128 + s * 16 + row_in_step;
        v[s] = Raw8<T>{};
        if (row < n) v[s] = load8<STREAM != kPlain>(w + static_cast<long long>(row) * k + kb * 128, part);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) amax = fmaxf(amax, abs_max8(to_f32(v[s])));
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) amax = fmaxf(amax, __shfl_xor(amax, d, 64));
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3])), 1e-4f);
    const float factor = kFp8Max / amax;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int row = nb * 128 + s * 16 + row_in_step;
        if (row < n)
            store_codes8<T, STREAM == kStreamBoth>(q + static_cast<long long>(row) * k + kb * 128, part, quantise8(to_f32(v[s]), factor));
    }
    if (threadIdx.x == 0) scales[static_cast<long long>(nb) * k_blocks + kb] = amax / kFp8Max;
}

// x [m, k] -> q [m, k] e4m3, scales fp32 with element (i, kb) at i * stride_m + kb * stride_k.
template <typename T>
inline hipError_t launch_per_token_cast(const T* x, void* q, float* scales, long long stride_m, long long stride_k,
                                        int m, int k, hipStream_t stream) {
    if (m == 0 || k == 0) return hipSuccess;
    if (m < 0 || k < 0 || (k % 128) != 0 || stride_m < 0 || stride_k < 0) return hipErrorInvalidValue;
    if (!x || !q || !scales) return hipErrorInvalidValue;
    constexpr int UNROLL = 2;      // measured: 1 ties or is up to 2 % slower, 4 is 2 to 20 % slower (fewer workgroups in flight)
    // The kernel counts groups in 32 bits: 2^31 of them would be 512 GB of bf16, more than a device holds.
    const long long k_blocks = k / 128, groups = m * k_blocks;
    const bool by_rows = stride_m < stride_k;
    const long long blocks = by_rows ? ceil_div<long long>(m, 16 * UNROLL) * k_blocks : ceil_div<long long>(groups, 16 * UNROLL);
    if (groups >= (1ll << 31) || blocks >= (1ll << 31)) return hipErrorInvalidValue;
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, stream, x, static_cast<uint8_t*>(q), scales,
                           uint32_t(m), uint32_t(k_blocks), stride_m, stride_k);
        return hipGetLastError();
    };
    if (cast_stream(groups * 128, sizeof(T), true) == kPlain)
        return by_rows ? launch(per_token_cast_kernel<T, UNROLL, true, kPlain>) : launch(per_token_cast_kernel<T, UNROLL, false, kPlain>);
    return by_rows ? launch(per_token_cast_kernel<T, UNROLL, true, kStreamSource>) : launch(per_token_cast_kernel<T, UNROLL, false, kStreamSource>);
}

// w [n, k] -> q [n, k] e4m3, scales fp32 [ceil(n/128), k/128] row-major.
template <typename T>
inline hipError_t launch_per_block_cast(const T* w, void* q, float* scales, int n, int k, hipStream_t stream) {
    if (n == 0 || k == 0) return hipSuccess;
    if (n < 0 || k < 0 || (k % 128) != 0) return hipErrorInvalidValue;
    if (!w || !q || !scales) return hipErrorInvalidValue;
    const long long blocks = static_cast<long long>(ceil_div(n, 128)) * (k / 128);
    if (blocks >= (1ll << 31)) return hipErrorInvalidValue;
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, stream, w, static_cast<uint8_t*>(q), scales, n, k);
        return hipGetLastError();
    };
    switch (cast_stream(static_cast<long long>(n) * k, sizeof(T), false)) {
        case kPlain: return launch(per_block_cast_kernel<T, kPlain>);
        case kStreamSource: return launch(per_block_cast_kernel<T, kStreamSource>);
        default: return launch(per_block_cast_kernel<T, kStreamBoth>);
    }
}

} // namespace yan
