// fp32 products on the bf16 matrix cores: each operand split without loss into
// three bf16 terms, a = a1 + a2 + a3 (each the rounding of what the ones before
// leave); a product takes the six terms above 2^-26 of it, a1 b1, a1 b2, a2 b1,
// a2 b2, a1 b3 and a3 b1, accumulated in fp32.
//
// Valid while no operand exceeds 2^50 in magnitude and no sum is nonzero below
// 2^-60: operands below 2^-102 lose low bits to bf16's least exponent, which
// moves a sum by at most K 2^-84.  A tile that meets a larger operand, or ends
// with a smaller or a non-finite sum (as any infinity or NaN operand gives), is
// computed again on v_mfma_f32_32x32x2_f32 from global memory.
#pragma once

#include "pxs_common.h"

namespace pxs {

constexpr float kSplitHigh = 0x1p50f, kSplitLow = 0x1p-60f;

// Whether a finished sum tells that the tile has to be computed again.
__device__ __forceinline__ bool split_sum_odd(float v) {
    const float m = fabsf(v);
    return !(m == 0.0f || (m >= kSplitLow && m < INFINITY));
}

// The six terms' planes (of A and B), the smaller terms first.
constexpr int kSplitTermA[6] = {2, 0, 1, 1, 0, 0}, kSplitTermB[6] = {0, 2, 1, 0, 1, 0};

// Splits 4 values into the three planes' 8-byte pieces; hi follows the largest
// magnitude seen.
__device__ __forceinline__ void split4(const float4 & f, uint2 (&out)[3], float & hi) {
    const float v[4] = {f.x, f.y, f.z, f.w};
    uint32_t w[3][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float a = v[2 * i], b = v[2 * i + 1];
        hi = fmaxf(hi, fmaxf(fabsf(a), fabsf(b)));
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            uint32_t pk = pack_bf16x2(a, b);
            asm("" : "+v"(pk));  // one conversion, not one more to take the low half apart
            w[q][i] = pk;
            if (q < 2) {
                a = a - __builtin_bit_cast(float, pk << 16);
                b = b - __builtin_bit_cast(float, pk & 0xffff0000u);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) out[q] = make_uint2(w[q][0], w[q][1]);
}

} // namespace pxs
