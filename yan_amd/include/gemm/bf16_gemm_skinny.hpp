// Dense 16-bit GEMM for up to 64 activation rows on the kernel of weight_stream.hpp. Same contract as bf16_gemm.hpp (c[m,n] =
// a[m,k] @ b[n,k]^T, fp32 accumulate; yan/jit_kernels/cute_gemm.py:21-64): a K block of 128 bytes is two 16x16x32 MFMAs per atom, the
// first over the even chunks, the second over the odd ones. The tiled kernels give a workgroup at least 64 weight rows, which leaves
// most compute units idle where n is a few thousand. Which problems run it: get_weight_stream_dense_config in
// yan_amd/jit_kernels/heuristics.py.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include "weight_stream.hpp"

namespace yan {

// Whether the weight-streaming kernel can run a problem at all: whole 128-byte K blocks, 8-byte output runs.
__host__ __device__ constexpr bool dense_skinny_fits(int m, int n, int k, int tm) {
    return m > 0 && m <= 16 * tm && n > 0 && (n % 4) == 0 && k > 0 && k < (1 << 30) && (k % 64) == 0;
}

// m <= 16 * TM; `num_sms` > 0 caps the workgroups. hipErrorInvalidValue for sizes outside the kernel's reach.
template <typename Atom, typename Elem, int TM>
inline hipError_t launch_dense_skinny(int m, int n, int k, const void* a, const void* b, void* c, hipStream_t stream, int num_sms = 0) {
    if (m == 0 || n == 0) return hipSuccess;
    if (!dense_skinny_fits(m, n, k, TM) || !a || !b || !c) return hipErrorInvalidValue;
    if (!launch_weight_stream<Atom, Elem, 0, 0, TM, kDense>(a, nullptr, 0, 0, b, nullptr, c, m, n, k * 2, num_sms, stream)) return hipErrorInvalidValue;
    return hipGetLastError();
}

} // namespace yan
