// Float32 products on the bfloat16 matrix units: each operand as the sum of three bfloat16, six of their nine products
// on v_mfma_f32_16x16x32_bf16, which together take 6/16 of v_mfma_f32_16x16x4_f32's time. The three parts hold a
// float32 from 2^-110 on exactly and the products left out (m.l, l.m, l.l) are below 2^-25 of h.h, so what rounds a
// result is, as there, the float32 accumulation, once per 32 k and product instead of once per 4 k. Measured against
// float64 (67200 x 256 x 256 normal operands): relative error 1.6e-7, against 2.0e-7 on the float32 units.
// Values that the split cannot take are noticed (SplitRange): infinite or so large that their bfloat16 may round to
// infinity (infinity - infinity is not what the product is), and so small that the parts fall under bfloat16's smallest
// subnormal, 2^-133 (relative error 2e-3 at 2^-126, with no bit left at 2^-140). The kernels compute what those touch
// on the float32 units instead.
#pragma once

#include "td_gemm.h"

namespace td {

typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));

// x = h + m + l, each a bfloat16 (24 significant bits in 8 + 8 + 8, round to nearest): exactly where SplitRange agrees
__device__ __forceinline__ void split3(f32x4 x, bf16x4& h, bf16x4& m, bf16x4& l) {
    h = __builtin_convertvector(x, bf16x4);
    const f32x4 r = x - __builtin_convertvector(h, f32x4);
    m = __builtin_convertvector(r, bf16x4);
    l = __builtin_convertvector(r - __builtin_convertvector(m, f32x4), bf16x4);
}

// Whether a value is non-finite, at least 2^127 in magnitude, or less than 2^-110 and not 0: two instructions a value
struct SplitRange {
    float hi = 0.f;            // the largest magnitude, NaN once one was seen
    unsigned lo = 0xffffffffu;  // the least of twice a value's bits (without its sign) less 1: 0 wraps to the largest
    __device__ __forceinline__ void add(f32x4 x) {
        const u32x4 u = __builtin_bit_cast(u32x4, x);
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
            hi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(hi, __builtin_fabsf(x[e])),
                                               __builtin_fabsf(x[e + 1]));
            lo = min(min(lo, (u[e] << 1) - 1u), (u[e + 1] << 1) - 1u);
        }
    }
    __device__ __forceinline__ bool beyond() const {
        return !(hi < 0x1p127f) || lo < (unsigned{127 - 110} << 24) - 1u;
    }
};

// The products of split operands in the order they are accumulated, small ones first: part of the first and of the
// second operand (0 h, 1 m, 2 l)
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0}, kSplitB[6] = {0, 2, 1, 0, 1, 0};

// A 128 x 128 tile of a split product by 2 x 2 wavefronts of 64 x 64: both operands' slices for 32 k in LDS, three
// planes of 128 rows of 64 bytes each. Row n lies at split_row(n), its chunk c of 8 k at slot c ^ (bits 1 and 2 of
// that): the 16 rows of a fragment read go at the full LDS rate, and so do stores of 8 bytes a row to every fourth row.
constexpr int kSplitTile = 128, kSplitPlane = kSplitTile * 32;
struct SplitSlices {
    bf16 a[3 * kSplitPlane], b[3 * kSplitPlane];
    int flags[4];  // a wavefront staged a value beyond the split's range
};
__device__ __forceinline__ int split_row(int n) { return n ^ ((n >> 2) & 3); }
__device__ __forceinline__ int split_at(int n, int chunk) {
    const int row = split_row(n);
    return row * 32 + (chunk ^ ((row >> 1) & 3)) * 8;
}

// acc[i][j] += a's rows 64 wa + 16 i .. times b's rows 64 wb + 16 j .. over the slices' 32 k: element e of acc[i][j] is
// a row 64 wa + 16 i + 4 (lane / 16) + e, b row 64 wb + 16 j + lane % 16. The 32 k's products are summed apart and then
// added: a long sum is rounded once per 32 k instead of six times (weight gradient of 67200 tokens: error against
// float64 4.2e-7 with them in one, 3.7e-7 on the float32 units).
__device__ __forceinline__ void split_mma(const SplitSlices& s, int wa, int wb, int lane, f32x4 (&acc)[4][4]) {
    const int at = split_at(lane & 15, lane >> 4);
    const bf16* const a = s.a + 64 * wa * 32 + at;
    const bf16* const b = s.b + 64 * wb * 32 + at;
    u32x4 fb[3][4];
#pragma unroll
    for (int o = 0; o < 3; ++o)
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[o][j] = *reinterpret_cast<const u32x4*>(b + o * kSplitPlane + 16 * j * 32);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        u32x4 fa[3];
#pragma unroll
        for (int o = 0; o < 3; ++o) fa[o] = *reinterpret_cast<const u32x4*>(a + o * kSplitPlane + 16 * i * 32);
        f32x4 t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) t[j] = KBlock<bf16>::mma(fa[kSplitA[q]], fb[kSplitB[q]][j], t[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += t[j];
    }
}

}  // namespace td
