// The ConvNeXt MLP of narrow levels in one kernel:
//   x += silu(LN(y) W0^T + b0) W2^T + b2        (src/slat_decoder.cpp:185-222)
// for y [rows, C] bf16 (the block's convolution), x fp32, W0 [M, C] and
// W2 [C, M] bf16.
//
// As separate launches the norm, the two linears and their [rows, M] hidden
// tensor are HBM passes: at 2.49M rows of 64 channels (M = 256) they moved 4.2
// GB where y, x and the result are 1.6 GB.  Here each wave keeps 32 rows in
// registers from y to the residual:
//   - lane (h, r) loads dims 16 t + 8 h .. + 7 of row r, which is the B operand
//     of K step t; the norm's sums are lane-local plus one exchange with the
//     partner lane, and its result goes back to the same registers as bf16;
//   - H^T = W0 Y^T: D's rows are hidden channels and its columns rows, so a
//     lane holds hidden channels of its own row r.  The W0 rows of a 32-channel
//     block are taken in the order hidden_row, so that registers 8 t .. 8 t + 7
//     are channels 16 t + 8 h .. + 7: after bias, SiLU and rounding they are the
//     B operand of K step t of the second product without leaving the lane;
//   - X^T += W2 H^T; a lane then updates 4 consecutive channels of its row.
// W0 and W2 stream through LDS in chunks of 64 hidden channels, two buffers,
// the next chunk's DMA in flight while one is multiplied; the 8 waves of a
// workgroup share them.
//
// Bound by the vector work between the two products (an exponential and a
// reciprocal per hidden value) more than by HBM.  At 256 channels the output's
// sums and the rows' operands take all 256 registers and 41 more spill.  Measured against the norm
// and the two linears: 2.68M rows of 64 channels 452 against 1,400 us, 671k of
// 128 394 against 812 us, 168k of 256 (M = 1024) 423 against 503 us.  Wider
// levels have few rows, and their output sums would not fit the registers.

#include "pxs_common.h"

namespace pxs {
namespace {

constexpr int kMlpWaves = 8, kMlpRows = kMlpWaves * 32, kMlpHidden = 64;
constexpr int kMlpMaxHidden = 1024;  // b0 in LDS

struct MlpArgs {
    const uint16_t * y;
    int64_t rows;
    float eps;
    const float * gamma;
    const float * beta;
    const uint16_t * w0;
    const float * b0;
    const uint16_t * w2;
    const float * b2;
    int hidden;
    const float * x_in;
    float * x_out;
};

// The hidden channel (of a block of 32) whose W0 row is the block's A-operand
// row i: i = 8 g + 4 h + e holds channel 16 (g / 2) + 8 h + 4 (g % 2) + e.
__device__ __forceinline__ int hidden_row(int i) {
    return (i & 16) | ((i & 4) << 1) | ((i & 8) >> 1) | (i & 3);
}

// XOR swizzle of the 16-byte pieces of a row of P pieces: the 16 rows that one
// LDS cycle of a fragment read serves land on different banks.
template <int P> __device__ __forceinline__ int mlp_swz(int row) {
    if constexpr (P == 8) return (row & 7) ^ ((row >> 3) & 1);
    else return row & 15;
}

__device__ __forceinline__ float silu_fast(float v) {
    // rounded to bf16 next: the hardware reciprocal's last-place error is lost in it
    return v * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(v * -1.4426950408889634f));
}

template <int C>
__global__ void __launch_bounds__(kMlpWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
convnext_mlp_kernel(MlpArgs a) {
    constexpr int KS = C / 16;               // K steps of the first product
    constexpr int OB = C / 32;               // 32-channel blocks of the output
    constexpr int P0 = C / 8;                // 16-byte pieces per W0 row
    constexpr int kW0 = kMlpHidden * C * 2;  // bytes of a W0 chunk; a W2 chunk is as large
    constexpr int kStage = 2 * kW0;
    constexpr int kInstr = kW0 / (1024 * kMlpWaves);  // DMA instructions per wave and operand
    static_assert(kInstr * 1024 * kMlpWaves == kW0, "chunk must split over the waves");
    extern __shared__ __align__(16) char smem[];
    float * bias0 = reinterpret_cast<float *>(smem + 2 * kStage);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r = lane & 31;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kMlpRows + wave * 32 + r;
    const bool live = row < a.rows;
    const int64_t src = live ? row : a.rows - 1;
    const uint32_t lds = lds_offset(smem);

    auto issue = [&](int chunk) __attribute__((always_inline)) {
        const uint32_t base = lds + (chunk & 1) * kStage;
#pragma unroll
        for (int j = 0; j < kInstr; ++j) {
            const int piece = (wave * kInstr + j) * 64 + lane;  // 16-byte piece of the chunk
            const int rw = piece / P0, slot = piece % P0;
            lds_dma16(a.w0 + static_cast<int64_t>(chunk * kMlpHidden + rw) * C + (slot ^ mlp_swz<P0>(rw)) * 8,
                      base + (wave * kInstr + j) * 1024);
        }
#pragma unroll
        for (int j = 0; j < kInstr; ++j) {
            const int piece = (wave * kInstr + j) * 64 + lane;
            const int rw = piece / 8, slot = piece % 8;
            lds_dma16(a.w2 + static_cast<int64_t>(rw) * a.hidden + chunk * kMlpHidden + (slot ^ mlp_swz<8>(rw)) * 8,
                      base + kW0 + (wave * kInstr + j) * 1024);
        }
    };

    for (int i = tid; i < a.hidden; i += kMlpWaves * 64) bias0[i] = a.b0 ? a.b0[i] : 0.0f;

    // The wave's rows and their norm.
    bf16x8 yf[KS];
    {
        uint4 raw[KS];
#pragma unroll
        for (int t = 0; t < KS; ++t)
            raw[t] = *reinterpret_cast<const uint4 *>(a.y + src * C + 16 * t + 8 * h);
        issue(0);
        auto unpack = [](const uint4 & u, float (&v)[8]) __attribute__((always_inline)) {
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
                v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
            }
        };
        float s = 0.0f;
#pragma unroll
        for (int t = 0; t < KS; ++t) {
            float v[8];
            unpack(raw[t], v);
#pragma unroll
            for (int e = 0; e < 8; ++e) s += v[e];
        }
        s += __shfl_xor(s, 32, 64);
        const float mean = s / static_cast<float>(C);
        float q = 0.0f;
#pragma unroll
        for (int t = 0; t < KS; ++t) {
            float v[8];
            unpack(raw[t], v);
#pragma unroll
            for (int e = 0; e < 8; ++e) q += (v[e] - mean) * (v[e] - mean);
        }
        q += __shfl_xor(q, 32, 64);
        const float inv = 1.0f / sqrtf(q / static_cast<float>(C) + a.eps);
#pragma unroll
        for (int t = 0; t < KS; ++t) {
            float v[8];
            unpack(raw[t], v);
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int c = 16 * t + 8 * h + 4 * i;
                const float4 g = *reinterpret_cast<const float4 *>(a.gamma + c);
                const float4 b = *reinterpret_cast<const float4 *>(a.beta + c);
                w[2 * i] = pack_bf16x2((v[4 * i] - mean) * inv * g.x + b.x, (v[4 * i + 1] - mean) * inv * g.y + b.y);
                w[2 * i + 1] = pack_bf16x2((v[4 * i + 2] - mean) * inv * g.z + b.z,
                                           (v[4 * i + 3] - mean) * inv * g.w + b.w);
            }
            yf[t] = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
        }
    }

    f32x16 out[OB];
#pragma unroll
    for (int o = 0; o < OB; ++o)
#pragma unroll
        for (int v = 0; v < 16; ++v) out[o][v] = 0.0f;

    const int chunks = a.hidden / kMlpHidden;
    const int hr = hidden_row(r);
    for (int c = 0; c < chunks; ++c) {
        wait_vmcnt(0);
        barrier_no_fence();  // chunk c (and bias0) in LDS; every wave is done with chunk c - 1
        if (c + 1 < chunks) issue(c + 1);
        const char * w0 = smem + (c & 1) * kStage;
        const char * w2 = w0 + kW0;
#pragma unroll
        for (int b = 0; b < kMlpHidden / 32; ++b) {
            f32x16 acc;
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
            const int wr = b * 32 + hr;
#pragma unroll
            for (int t = 0; t < KS; ++t) {
                const bf16x8 wf = *reinterpret_cast<const bf16x8 *>(
                    w0 + wr * (C * 2) + (((2 * t + h) ^ mlp_swz<P0>(wr)) << 4));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, yf[t], acc, 0, 0, 0);
            }
            bf16x8 hf[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                uint32_t w[4];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float4 bv = *reinterpret_cast<const float4 *>(
                        bias0 + c * kMlpHidden + b * 32 + 16 * t + 8 * h + 4 * i);
                    const int v = 8 * t + 4 * i;
                    w[2 * i] = pack_bf16x2(silu_fast(acc[v] + bv.x), silu_fast(acc[v + 1] + bv.y));
                    w[2 * i + 1] = pack_bf16x2(silu_fast(acc[v + 2] + bv.z), silu_fast(acc[v + 3] + bv.w));
                }
                hf[t] = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int o = 0; o < OB; ++o) {
                    const int rw = o * 32 + r;
                    const bf16x8 wf = *reinterpret_cast<const bf16x8 *>(
                        w2 + rw * 128 + (((4 * b + 2 * t + h) ^ mlp_swz<8>(rw)) << 4));
                    out[o] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, hf[t], out[o], 0, 0, 0);
                }
        }
    }
    if (!live) return;
#pragma unroll
    for (int o = 0; o < OB; ++o)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int c = o * 32 + 8 * g + 4 * h;
            float4 v = *reinterpret_cast<const float4 *>(a.x_in + row * C + c);
            float4 b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (a.b2) b = *reinterpret_cast<const float4 *>(a.b2 + c);
            v.x += out[o][4 * g] + b.x;
            v.y += out[o][4 * g + 1] + b.y;
            v.z += out[o][4 * g + 2] + b.z;
            v.w += out[o][4 * g + 3] + b.w;
            *reinterpret_cast<float4 *>(a.x_out + row * C + c) = v;
        }
}

template <int C>
int launch_mlp(const MlpArgs & a, hipStream_t s) {
    constexpr int smem = 4 * kMlpHidden * C * 2 + kMlpMaxHidden * 4;
    if constexpr (smem > 64 * 1024) {
        static bool configured = false;
        if (!configured) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&convnext_mlp_kernel<C>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, smem);
            if (e != hipSuccess) return check_hip(e, "hipFuncSetAttribute(convnext_mlp)");
            configured = true;
        }
    }
    hipLaunchKernelGGL(convnext_mlp_kernel<C>, dim3(grid_for(a.rows, kMlpRows)), dim3(kMlpWaves * 64), smem, s, a);
    return check_launch("ConvNeXt MLP");
}

bool aligned16(const void * p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

} // namespace

int convnext_mlp(const void * y, int64_t rows, int channels, float eps, const float * gamma,
                 const float * beta, const void * w0, const float * b0, const void * w2,
                 const float * b2, int hidden, const float * x_in, float * x_out, hipStream_t s,
                 bool * done) {
    *done = false;
    if (hidden % kMlpHidden != 0 || hidden > kMlpMaxHidden || !aligned16(y) || !aligned16(gamma) ||
        !aligned16(beta) || !aligned16(w0) || !aligned16(w2) || !aligned16(b2) || !aligned16(x_in) ||
        !aligned16(x_out) || rows > static_cast<int64_t>(INT32_MAX) * kMlpRows)
        return PXS_OK;
    const MlpArgs a{static_cast<const uint16_t *>(y), rows, eps, gamma, beta,
                    static_cast<const uint16_t *>(w0), b0, static_cast<const uint16_t *>(w2), b2, hidden,
                    x_in, x_out};
    *done = true;
    // A workgroup walks the whole hidden width for its 256 rows, so a call of few
    // rows takes as long as one that fills the CUs, and the separate launches, which
    // split the columns too, are done sooner.  The whole block, us, in one kernel
    // against the separate launches, M = 4 C: 64 channels at 300 rows 38 / 45 (M =
    // 1024 54 / 52); 128 at 1,000 rows 78 / 71, 4,096 78 / 75, 8,000 81 / 84, 20,000 85 /
    // 101; 256 at 1,000 rows 232 / 153, 20,000 248 / 203, 32,768 (half the CUs) 265 /
    // 250, 35,000 373 / 380, 50,000 397 / 436.
    if (channels == 64 && (hidden <= 512 || rows >= 4096)) return launch_mlp<64>(a, s);
    if (channels == 128 && rows >= 8192) return launch_mlp<128>(a, s);
    if (channels == 256 && rows > 32768) return launch_mlp<256>(a, s);
    *done = false;
    return PXS_OK;
}

} // namespace pxs
