// fp32 products on the bf16 matrix cores: each operand split without loss into
// three bf16 terms, a = a1 + a2 + a3 (each the rounding of what the ones before
// leave); a product takes the six terms above 2^-26 of it, a1 b1, a1 b2, a2 b1,
// a2 b2, a1 b3 and a3 b1, accumulated in fp32.
//
// Range.  Operands below 2^-110 lose bits under bf16's least step, 2^-133, at
// most 2^-134 each, which moves a sum of K products with operands up to hi by at
// most 2 K hi 2^-134 (the matrix instruction keeps subnormal operands, products
// and sums).  So a sum of magnitude K max(hi, 2^-15) 2^-109 and more is within
// 2^-24 of itself of the same sum of whole operands; no operand may exceed 2^50.
// An output that ends smaller, or not finite (as any infinity or NaN operand
// makes it), or zero though its row or channel holds operands below 2^-110, is
// taken again on v_mfma_f32_32x32x2_f32 from global memory.  Whether it is, and so
// its bits, depend on its own operands only (and, in a convolution, on the weights
// of offsets that only other rows of its tile have).  Kernels look in two steps: ordinary
// tiles pay for one comparison per sum with the bound of hi = 2^50; a tile with
// smaller sums takes its own hi, and looks for small operands where sums are zero.
// Measured, us, ordinary inputs first: linear 20,000 x 1024 -> 1024 242, scaled by
// 1e-20 243, by 1e-26 (some sums near zero in most tiles) 690, an infinity in every
// tile 970, a row of zeros in every tile 253, zero weights 350; convolution of 30,000
// rows 64 -> 64 80, by 1e-20 85, an infinity in every tile 220, half the rows zero 120;
// attention of 4,000 x 16 heads 370, values by 1e-20 371, an infinite value 1,795, zero
// columns 378.
#pragma once

#include "pxs_common.h"

namespace pxs {

constexpr float kSplitHigh = 0x1p50f, kSplitWhole = 0x1p-110f;

// The least magnitude of a sum of `terms` products of operands up to hi.
__device__ __forceinline__ float split_low(float hi, int terms) {
    return fmaxf(hi, 0x1p-15f) * (static_cast<float>(terms) * 0x1p-109f);
}

// Whether a finished sum may have to be taken again (zero is looked at later).
__device__ __forceinline__ bool split_sum_odd(float v, float low) {
    const float m = fabsf(v);
    return !((m >= low) & (m < INFINITY));
}

// Whether an output with the operands' largest magnitude hi has to be; small: one
// of them is nonzero and below kSplitWhole.
__device__ __forceinline__ bool split_again(float v, float hi, bool small, int terms) {
    const bool zero = v == 0.0f;
    return (hi > kSplitHigh) | (zero & small) | (!zero & split_sum_odd(v, split_low(hi, terms)));
}

__device__ __forceinline__ bool split_small(float v) { return (v != 0.0f) & (fabsf(v) < kSplitWhole); }
__device__ __forceinline__ bool split_small(const float4 & f) {
    return split_small(f.x) | split_small(f.y) | split_small(f.z) | split_small(f.w);
}
__device__ __forceinline__ float max_abs(const float4 & f) {
    return fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fmaxf(fabsf(f.z), fabsf(f.w)));
}

// The largest v (>= 0) of the workgroup, through one word of LDS that no wave
// uses any more.
__device__ __forceinline__ float split_block_max(float v, uint32_t * word) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    if (threadIdx.x == 0) *word = 0u;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) atomicMax(word, __builtin_bit_cast(uint32_t, v));
    __syncthreads();
    return __builtin_bit_cast(float, *word);
}

// The outputs of one wave's 32 x 32 block that split_again names, from a second
// sum taken on v_mfma_f32_32x32x2_f32: A's row r in lane r (and r + 32), B's
// likewise, hi_a, hi_b, small_a and small_b of the K that the lane has read.
// Register v of D is A's row 8 (v / 4) + 4 h + v % 4, lane r B's row r.
__device__ __forceinline__ void split_select(float (&sum)[16], const f32x16 & second, float hi_a, float hi_b,
                                             bool small_a, bool small_b, int terms, int h) {
    hi_a = fmaxf(hi_a, __shfl_xor(hi_a, 32, 64));
    hi_b = fmaxf(hi_b, __shfl_xor(hi_b, 32, 64));
    int sa = small_a ? 1 : 0, sb = small_b ? 1 : 0;
    sa |= __shfl_xor(sa, 32, 64);
    sb |= __shfl_xor(sb, 32, 64);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = 8 * (v >> 2) + 4 * h + (v & 3);
        const float hi = fmaxf(__shfl(hi_a, row, 64), hi_b);
        const int small = __shfl(sa, row, 64) | sb;
        // (on plain floats and without branches: as an if on an element of a vector the
        // compiler, clang of ROCm 7.2, left the copy out, and whole vectors spilled)
        sum[v] = split_again(sum[v], hi, small != 0, terms) ? second[v] : sum[v];
    }
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
