// Block-scaled FP8 GEMM for up to 64 activation rows on the kernel of weight_stream.hpp. Same contract as fp8_gemm.hpp (operands of
// yan/jit_kernels/gemm.py:23-30, scale granularity of yan/include/gemm/fp8_gemm.cuh:48-61): per K block one 16x16x128 MFMA
// per atom from a zero accumulator, folded in with acc += p * (sA * sB) as the tiled kernel does. Which problems run it:
// get_weight_stream_fp8_config in yan_amd/jit_kernels/heuristics.py.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include "weight_stream.hpp"

namespace yan {

// m <= 16 * TM; `num_sms` > 0 caps the workgroups. hipErrorInvalidValue for sizes outside the kernel's reach.
template <int SHAPE_N, int SHAPE_K, int TM>
inline hipError_t launch_fp8_skinny(__hip_bfloat16* out, const void* lhs, const float* lhs_scales, int lhs_scales_stride_m,
                                    int lhs_scales_stride_k, const void* rhs, const float* rhs_scales, int m, int n, int k,
                                    hipStream_t stream, int num_sms = 0) {
    if (m == 0 || n == 0) return hipSuccess;
    if (m < 0 || m > 16 * TM || n < 0 || k <= 0 || (n % 4) != 0 || (k % 128) != 0) return hipErrorInvalidValue;
    if ((SHAPE_N && n != SHAPE_N) || (SHAPE_K && k != SHAPE_K)) return hipErrorInvalidValue;
    if (!out || !lhs || !lhs_scales || !rhs || !rhs_scales) return hipErrorInvalidValue;
    if (!launch_weight_stream<MfmaFP8_16x16x128, __bf16, SHAPE_N, SHAPE_K, TM, kScaled>(lhs, lhs_scales, lhs_scales_stride_m, lhs_scales_stride_k, rhs,
                                                                                   rhs_scales, out, m, n, k, num_sms, stream)) return hipErrorInvalidValue;
    return hipGetLastError();
}

// bf16 activations, quantised as launch_per_token_cast does it in every workgroup: A_ROWS is cast_rows(m, k / 128).
template <int SHAPE_N, int SHAPE_K, int A_ROWS>
inline hipError_t launch_fp8_skinny_cast(__hip_bfloat16* out, const void* x, const void* rhs, const float* rhs_scales, int m, int n, int k,
                                         hipStream_t stream, int num_sms = 0) {
    if (m == 0 || n == 0) return hipSuccess;
    if (m < 0 || n < 0 || k <= 0 || cast_rows(m, k / 128) != A_ROWS || (n % 4) != 0 || (k % 128) != 0) return hipErrorInvalidValue;
    if ((SHAPE_N && n != SHAPE_N) || (SHAPE_K && k != SHAPE_K)) return hipErrorInvalidValue;
    if (!out || !x || !rhs || !rhs_scales) return hipErrorInvalidValue;
    if (!launch_weight_stream<MfmaFP8_16x16x128, __bf16, SHAPE_N, SHAPE_K, 1, kCast, A_ROWS>(x, nullptr, 0, 0, rhs, rhs_scales, out, m, n, k, num_sms,
                                                                                           stream)) return hipErrorInvalidValue;
    return hipGetLastError();
}

} // namespace yan
