// Float32 products on the bfloat16 matrix units: each operand as the sum of three bfloat16, six of their nine products
// on v_mfma_f32_16x16x32_bf16, which together take 6/16 of v_mfma_f32_16x16x4_f32's time. The three parts hold a
// float32 exactly and the products left out (m.l, l.m, l.l) are below 2^-25 of h.h, so what rounds a result is, as
// there, the float32 accumulation, once per 32 k and product instead of once per 4 k. Measured against float64
// (67200 x 256 x 256 normal operands): relative error 1.6e-7, against 2.0e-7 on the float32 units.
// Values that the split cannot take (non-finite, or so large that their bfloat16 may round to infinity, and infinity
// - infinity is not what the product is) are noticed by beyond_split; the kernels compute what they touch by float32
// FMAs instead.
#pragma once

#include "td_gemm.h"

namespace td {

typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));

// x = h + m + l exactly, each a bfloat16 (24 significant bits in 8 + 8 + 8, round to nearest)
__device__ __forceinline__ void split3(f32x4 x, bf16x4& h, bf16x4& m, bf16x4& l) {
    h = __builtin_convertvector(x, bf16x4);
    const f32x4 r = x - __builtin_convertvector(h, f32x4);
    m = __builtin_convertvector(r, bf16x4);
    l = __builtin_convertvector(r - __builtin_convertvector(m, f32x4), bf16x4);
}

// whether a component is non-finite or at least 2^127 in magnitude
__device__ __forceinline__ bool beyond_split(f32x4 x) {
    const u32x4 u = __builtin_bit_cast(u32x4, x);
    const unsigned a = max(u[0] << 1, u[1] << 1), b = max(u[2] << 1, u[3] << 1);
    return max(a, b) >= 0xfe000000u;
}

// The products of split operands in the order they are accumulated, small ones first: part of the first and of the
// second operand (0 h, 1 m, 2 l)
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0}, kSplitB[6] = {0, 2, 1, 0, 1, 0};

}  // namespace td
