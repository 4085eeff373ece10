// Dense GEMM on MFMA for the plain linears: sparse_linear / varlen_linear
// (src/sparse.cpp:337-488) and the transformer block's gated and residual
// linears (src/sparse_transformer.cpp:229-235), in bf16 or fp32.
//
//   Y[m, n] = sum_k X[m, k] W[n, k] + bias[n]   then one epilogue:
//     store        y[m, n] = act(Y)                 (y in the operands' dtype)
//     add residual r[m, n] = r[m, n] + Y            (r fp32)
//     gate         r[m, n] = r[m, n] + Y * (block_mod[o + n] + time_mod[b(m), o + n])
//
// X rows and W rows are both contiguous along K, so a workgroup's BM x BN
// output tile streams 128-byte K chunks of BM rows of X and BN rows of W
// from L2 into LDS with global_load_lds_dwordx4 (no VGPR staging, no row
// map), two chunks in flight.  The loads use the instruction's scalar-base
// form: the tile's base address advances by 128 bytes per chunk in SGPRs and
// every lane keeps one fixed 32-bit offset per instruction, so the K loop
// issues no vector address arithmetic.  Rows past the end of X or W are
// clamped to the last row (valid memory; their outputs are not stored).
//
// MFMA operands are swapped relative to the output: the W fragment is the
// instruction's A operand and the X fragment its B operand, so D = Y^T per
// 32 x 32 block and lane (h, r) holds output row r, channels 8g + 4h + 0..3
// for g = 0..3: four consecutive channels per lane.
//   bf16: v_mfma_f32_32x32x16_bf16, 4 K steps of 16 per chunk (dense_gemm_kernel);
//   fp32: the same instruction on operands split in three (dense_split_kernel).
// The K order inside a chunk is permuted identically for both operands so a
// lane reads 16 contiguous bytes per LDS access; pieces are XOR-swizzled by
// row so the 16 rows one LDS cycle serves read 16 different bank groups.
// The fragments of K step u + 1 are read while step u multiplies.
//
// Plain stores go through LDS (each wave's block is written there and read
// back as whole 16-byte row pieces, so a store instruction covers 128-byte
// row segments); the residual forms read, add and write 4 channels per lane.
// Tile shapes (measured on MI355X against hipBLASLt's 256 x 256 kernels on
// the flow block's, the window workload's and the decoder's shapes):
//   256 x 256, 16 waves of 64 x 64, each wave issuing its share of the next
//     chunk's DMA one part per K step (one instruction burst per chunk left
//     the vector-memory return path idle between chunks);
//   128 x 128, 8 waves of 64 x 32 (two workgroups per CU);
//   128 x 64, 4 waves of 64 x 32 (three workgroups per CU; 64 outputs);
// chosen per shape by the number of rounds of tiles over the 256 CUs.

#include "pxs_common.h"
#include "split3.h"

#include <algorithm>

namespace pxs {
namespace {

enum DenseEpi { kDenseStore = 0, kDenseAddResidual = 1, kDenseGate = 2, kDensePartial = 3 };

struct DenseArgs {
    const void * x;        // [m, k]
    const void * w;        // [n, k]
    const float * bias;    // [n] or null
    int64_t m;
    int k;
    int n;
    void * y;              // [m, n], store epilogue
    int act;
    float * residual;      // [m, n] fp32, residual epilogues
    const int32_t * coords;      // [m, 4], gate epilogue: batch of each row
    const float * block_mod;     // gate = block_mod[gate_offset + c] + time_mod[b, gate_offset + c]
    const float * time_mod;      // [batch, 6 n]
    int gate_offset;
    int vec_out;           // 1: 4-channel vector accesses; 2: also whole 16-byte row pieces
    int group_m;           // tile order: groups of group_m row tiles, each walked down its rows first
    int splits;            // kDensePartial: K split over gridDim.y, sums to residual[split][m][n]
};

// Linears of one input with several weights: output g is at y + g m n.
struct DenseGroup {
    const void * w[kDenseGroup];
    const float * bias[kDenseGroup];
};
template <typename T> __device__ __forceinline__ void select_group(DenseArgs & a, const DenseGroup & g) {
    a.w = g.w[blockIdx.y];
    a.bias = g.bias[blockIdx.y];
    a.y = static_cast<T *>(a.y) + static_cast<int64_t>(blockIdx.y) * a.m * a.n;
}

// Output tile (row tile, column tile) of logical tile t: groups of g row
// tiles share their column tiles, and inside a group consecutive t walk the
// rows, so the tiles one XCD runs at a time cover g row tiles x (32 / g)
// column tiles of operands instead of one row tile x every column tile.
__device__ __forceinline__ void tile_of(int t, int tiles_m, int tiles_n, int g, int & tm, int & tn) {
    if (g <= 1) {
        tm = t / tiles_n;
        tn = t % tiles_n;
        return;
    }
    const int per_group = g * tiles_n;
    const int grp = t / per_group, in = t % per_group;
    const int rows = min(g, tiles_m - grp * g);  // the last group may be short
    tm = grp * g + in % rows;
    tn = in / rows;
}

__device__ __align__(16) uint4 g_dense_zero[8];  // 128 zero bytes: K pieces past the end

template <typename T> struct Store4;
template <> struct Store4<uint16_t> {
    static __device__ __forceinline__ void put(uint16_t * p, const float (&v)[4]) {
        uint2 u;
        u.x = pack_bf16x2(v[0], v[1]);
        u.y = pack_bf16x2(v[2], v[3]);
        *reinterpret_cast<uint2 *>(p) = u;
    }
};
template <> struct Store4<float> {
    static __device__ __forceinline__ void put(float * p, const float (&v)[4]) {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    }
};

// Epilogue of one wave: acc[i][j] is the 32 x 32 block (rows i, channels j);
// lane (h, r) holds row r and channels 8 g + 4 h + e at acc[i][j][4 g + e].
// The per-element arithmetic is the gather-GEMM epilogue's (value = acc +
// bias, then the activation; residual + value; residual + value * gate).
template <typename T, int TI, int TJ, int EPI>
__device__ __forceinline__ void dense_epilogue(const DenseArgs & a, const f32x16 (&acc)[TI][TJ],
                                               int64_t row0, int col0, int h, int r) {
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const int64_t row = row0 + i * 32 + r;
        if (row >= a.m) continue;
        int batch = 0;
        if constexpr (EPI == kDenseGate) batch = a.coords[row * 4];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = col0 + j * 32 + 8 * g + 4 * h;
                if (c >= a.n) continue;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e];
                if constexpr (EPI == kDensePartial) {
                    // cout is a multiple of 4 (dense_splits)
                    *reinterpret_cast<float4 *>(a.residual + row * a.n + c) = make_float4(v[0], v[1], v[2], v[3]);
                } else if (a.vec_out && c + 3 < a.n) {
                    if (a.bias) {
                        const float4 b = *reinterpret_cast<const float4 *>(a.bias + c);
                        v[0] = v[0] + b.x; v[1] = v[1] + b.y; v[2] = v[2] + b.z; v[3] = v[3] + b.w;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = v[e] + 0.0f;
                    }
                    if constexpr (EPI == kDenseStore) {
                        if (a.act == PXS_ACT_GELU_TANH) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_f(v[e]);
                        } else if (a.act == PXS_ACT_SILU) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[e] = silu_f(v[e]);
                        }
                        Store4<T>::put(static_cast<T *>(a.y) + row * a.n + c, v);
                    } else if constexpr (EPI == kDenseAddResidual) {
                        float4 * res = reinterpret_cast<float4 *>(a.residual + row * a.n + c);
                        float4 o = *res;
                        o.x = o.x + v[0]; o.y = o.y + v[1]; o.z = o.z + v[2]; o.w = o.w + v[3];
                        *res = o;
                    } else {
                        const float4 bm = *reinterpret_cast<const float4 *>(a.block_mod + a.gate_offset + c);
                        const float4 tm = *reinterpret_cast<const float4 *>(
                            a.time_mod + static_cast<int64_t>(batch) * 6 * a.n + a.gate_offset + c);
                        float4 * res = reinterpret_cast<float4 *>(a.residual + row * a.n + c);
                        float4 o = *res;
                        o.x = o.x + v[0] * (bm.x + tm.x);
                        o.y = o.y + v[1] * (bm.y + tm.y);
                        o.z = o.z + v[2] * (bm.z + tm.z);
                        o.w = o.w + v[3] * (bm.w + tm.w);
                        *res = o;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int ce = c + e;
                        if (ce >= a.n) break;
                        float val = v[e] + (a.bias ? a.bias[ce] : 0.0f);
                        if constexpr (EPI == kDenseStore) {
                            if (a.act == PXS_ACT_GELU_TANH) val = gelu_tanh_f(val);
                            else if (a.act == PXS_ACT_SILU) val = silu_f(val);
                            store_f32(static_cast<T *>(a.y) + row * a.n + ce, val);
                        } else if constexpr (EPI == kDenseAddResidual) {
                            float * res = a.residual + row * a.n + ce;
                            *res = *res + val;
                        } else {
                            const float gate = a.block_mod[a.gate_offset + ce] +
                                               a.time_mod[static_cast<int64_t>(batch) * 6 * a.n +
                                                          a.gate_offset + ce];
                            float * res = a.residual + row * a.n + ce;
                            *res = *res + val * gate;
                        }
                    }
                }
            }
        }
    }
}

// Row pitch in LDS of a wave's block in the staged store epilogue: 16 bytes
// of padding keep the 32 rows one fragment write covers on distinct banks
// (two-way at most).
template <typename T, int WN> constexpr int staged_pitch() { return WN * static_cast<int>(sizeof(T)) + 16; }

// Store epilogue through LDS: each wave writes its WM x WN block (bias and
// activation applied, rounded to T) into its own LDS region, then reads it
// back row by row, 16 contiguous bytes per lane, so every store instruction
// covers whole 128-byte row segments instead of 16 bytes in each of 32 rows.
// Same per-element arithmetic as dense_epilogue.  Needs n a multiple of 16 /
// sizeof(T) and y 16-byte aligned (vec_out with that n).
template <typename T, int TI, int TJ>
__device__ __forceinline__ void dense_store_staged(const DenseArgs & a, const f32x16 (&acc)[TI][TJ],
                                                   char * region, int64_t row0, int col0, int h,
                                                   int r, int lane) {
    constexpr int WM = TI * 32, WN = TJ * 32;
    constexpr int kPitch = staged_pitch<T, WN>();
    constexpr int kRowBytes = WN * static_cast<int>(sizeof(T));
    constexpr int kLanesPerRow = kRowBytes / 16;
    constexpr int kRowsPerPass = 64 / kLanesPerRow;
    constexpr int kElems = 16 / static_cast<int>(sizeof(T));
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int cl = j * 32 + 8 * g + 4 * h;  // column inside the block
            const int c = col0 + cl;
            float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (a.bias && c < a.n) {
                const float4 bv = *reinterpret_cast<const float4 *>(a.bias + c);
                b[0] = bv.x; b[1] = bv.y; b[2] = bv.z; b[3] = bv.w;
            }
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = acc[i][j][4 * g + e] + b[e];
                    if (a.act == PXS_ACT_GELU_TANH) v[e] = gelu_tanh_f(v[e]);
                    else if (a.act == PXS_ACT_SILU) v[e] = silu_f(v[e]);
                }
                Store4<T>::put(reinterpret_cast<T *>(region + (i * 32 + r) * kPitch + cl * sizeof(T)), v);
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's own writes are in LDS
    const int lr = lane / kLanesPerRow, lc = lane % kLanesPerRow;
#pragma unroll
    for (int pass = 0; pass < WM / kRowsPerPass; ++pass) {
        const int rl = pass * kRowsPerPass + lr;
        const int64_t row = row0 + rl;
        const uint4 v = *reinterpret_cast<const uint4 *>(region + rl * kPitch + lc * 16);
        const int c = col0 + lc * kElems;
        if (row < a.m && c < a.n)
            *reinterpret_cast<uint4 *>(static_cast<T *>(a.y) + row * a.n + c) = v;
    }
}

// Rows of KB = 128 bytes per K chunk in LDS: 8 pieces of 16 bytes,
// XOR-swizzled by row so that the 16 rows one LDS cycle serves (64 banks of
// 4 bytes) read 16 different bank groups.
template <int KB> __device__ __forceinline__ int piece_swz(int row);
template <> __device__ __forceinline__ int piece_swz<128>(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// Waits until at most min(later, MAX) stages of PER instructions each are in
// flight (s_waitcnt's count is a constant, six bits of it vmcnt).
template <int MAX, int PER>
__device__ __forceinline__ void wait_stages(int later) {
    constexpr int n = MAX * PER;
    static_assert(n < 64, "vmcnt has six bits");
    if constexpr (MAX > 0) {
        if (later < MAX) {
            wait_stages<MAX - 1, PER>(later);
            return;
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70 | (n & 15) | ((n >> 4) << 14));
}

// NW waves in a WAVES_M x (NW / WAVES_M) grid, each owning a (BM / WAVES_M) x
// (BN / WAVES_N) block of the tile; NSTAGE K chunks of KB bytes per row in
// flight (one DMA instruction fills 1 KiB: 1024 / KB rows).
// With a GROUP (DenseGroup) argument, blockIdx.y picks its weights, bias and output.
template <typename T, int BM, int BN, int NW, int WAVES_M, int NSTAGE, int KB, int EPI, bool SPREAD,
          bool STAGED, typename... GROUP>
__global__ void __launch_bounds__(NW * 64)
dense_gemm_kernel(DenseArgs a, GROUP... group) {
    constexpr int kVec = 16 / static_cast<int>(sizeof(T));  // elements per piece
    constexpr int P = KB / 16;                              // pieces per chunk row
    constexpr int kChunk = P * kVec;                        // elements per chunk row
    constexpr int RPI = 1024 / KB;                          // rows per DMA instruction
    constexpr int WAVES_N = NW / WAVES_M;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    constexpr int TI = WM / 32, TJ = WN / 32;
    static_assert(sizeof(T) == 2, "fp32 products run on dense_split_kernel");
    static_assert(TI * 32 * WAVES_M == BM && TJ * 32 * WAVES_N == BN, "wave blocks must tile");
    constexpr int kStage = (BM + BN) * KB;
    constexpr int AI = BM / (RPI * NW);  // DMA instructions per wave per stage
    constexpr int BI = BN / (RPI * NW);
    static_assert(AI * RPI * NW == BM && BI * RPI * NW == BN, "tile rows must split over the waves");
    constexpr int kPerStage = AI + BI;

    extern __shared__ __align__(16) char smem[];
    if constexpr (sizeof...(GROUP) > 0) select_group<T>(a, group...);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int h = lane >> 5, r = lane & 31;

    const int tiles_n = (a.n + BN - 1) / BN;
    const int tiles_m = static_cast<int>((a.m + BM - 1) / BM);
    const int logical = remap_xcd(blockIdx.x, gridDim.x);
    int tm, tn;
    tile_of(logical, tiles_m, tiles_n, a.group_m, tm, tn);
    const int64_t p0 = static_cast<int64_t>(tm) * BM;
    const int n0 = tn * BN;

    const char * xs = static_cast<const char *>(a.x) + p0 * a.k * static_cast<int64_t>(sizeof(T));
    const char * wsb = static_cast<const char *>(a.w) + static_cast<int64_t>(n0) * a.k * sizeof(T);
    // Stages of this workgroup: all of K, or its split's share of them.
    const int all_stages = (a.k + kChunk - 1) / kChunk;
    int stage0 = 0, stages = all_stages;
    if constexpr (EPI == kDensePartial) {
        stage0 = static_cast<int>(blockIdx.y) * all_stages / a.splits;
        stages = (static_cast<int>(blockIdx.y) + 1) * all_stages / a.splits - stage0;
        a.residual += static_cast<int64_t>(blockIdx.y) * a.m * a.n;
        xs += static_cast<int64_t>(stage0) * KB;
        wsb += static_cast<int64_t>(stage0) * KB;
    }
    const bool ragged = a.k % kChunk != 0;  // the last chunk of K holds pieces past k
    // Fixed per-lane parts of the loads: row lane / P of each instruction,
    // clamped into the operand, and the swizzled piece it fetches.
    const int lrow = lane / P, lslot = lane % P;
    const int64_t last_x = a.m - 1 - p0;
    const int last_w = a.n - 1 - n0;
    uint32_t a_off[AI], b_off[BI];
#pragma unroll
    for (int j = 0; j < AI; ++j) {
        const int row = (wave * AI + j) * RPI + lrow;
        const int64_t rr = row < last_x ? row : last_x;
        a_off[j] = static_cast<uint32_t>(rr * a.k * static_cast<int64_t>(sizeof(T)) +
                                         (lslot ^ piece_swz<KB>(row)) * 16);
    }
#pragma unroll
    for (int j = 0; j < BI; ++j) {
        const int row = (wave * BI + j) * RPI + lrow;
        const int rr = row < last_w ? row : last_w;
        b_off[j] = static_cast<uint32_t>(static_cast<int64_t>(rr) * a.k * sizeof(T) +
                                         (lslot ^ piece_swz<KB>(row)) * 16);
    }

    // DMA instruction q of stage s: q < AI fills X rows, the rest W rows.
    auto issue_one = [&](int s, int q) __attribute__((always_inline)) {
        char * base = smem + (s % NSTAGE) * kStage;
        const int64_t kb = static_cast<int64_t>(s) * KB;
        const bool is_x = q < AI;
        const int j = is_x ? q : q - AI;
        const int row = (wave * (is_x ? AI : BI) + j) * RPI + lrow;
        const uint32_t lds = lds_offset(base + ((is_x ? 0 : BM) + (wave * (is_x ? AI : BI) + j) * RPI) * KB);
        const char * src = is_x ? xs : wsb;
        const uint32_t off = is_x ? a_off[j] : b_off[j];
        if (ragged && stage0 + s == all_stages - 1) {
            // Pieces past k come from the zero line.
            const bool in = (stage0 + s) * kChunk + (lslot ^ piece_swz<KB>(row)) * kVec < a.k;
            lds_dma16(in ? static_cast<const void *>(src + kb + off) : static_cast<const void *>(g_dense_zero), lds);
        } else {
            lds_dma16_sbase(src + kb, off, lds);
        }
    };
    auto issue = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kPerStage; ++q) issue_one(s, q);
    };

    f32x16 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

#pragma unroll
    for (int s = 0; s < NSTAGE - 1; ++s)
        if (s < stages) issue(s);

    for (int s = 0; s < stages; ++s) {
        wait_stages<NSTAGE - 2, kPerStage>(stages - 1 - s);
        barrier_no_fence();
        const bool more = s + NSTAGE - 1 < stages;
        if (!SPREAD && more) issue(s + NSTAGE - 1);
        const char * sx = smem + (s % NSTAGE) * kStage;
        const char * sw = sx + BM * KB;
        // Half h of the wave's lanes reads pieces (P / 2) h .. (P / 2) h + P / 2 - 1;
        // the fragments of K step u + 1 are read while step u multiplies.
        uint4 xr[2][TI], wr[2][TJ];
        auto read_frags = [&](int u, uint4 (&xo)[TI], uint4 (&wo)[TJ]) __attribute__((always_inline)) {
            const int piece = (P / 2) * h + u;
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                const int row = wm * WM + i * 32 + r;
                xo[i] = *reinterpret_cast<const uint4 *>(sx + row * KB + ((piece ^ piece_swz<KB>(row)) << 4));
            }
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                const int row = wn * WN + j * 32 + r;
                wo[j] = *reinterpret_cast<const uint4 *>(sw + row * KB + ((piece ^ piece_swz<KB>(row)) << 4));
            }
        };
        read_frags(0, xr[0], wr[0]);
#pragma unroll
        for (int u = 0; u < P / 2; ++u) {
            if constexpr (SPREAD) {
                // The next stage's DMA in P / 2 parts, one per K step.
#pragma unroll
                for (int q = 0; q < kPerStage; ++q)
                    if (more && q * (P / 2) / kPerStage == u) issue_one(s + NSTAGE - 1, q);
            }
            if (u + 1 < P / 2) read_frags(u + 1, xr[(u + 1) & 1], wr[(u + 1) & 1]);
            const uint4 (&xc)[TI] = xr[u & 1];
            const uint4 (&wc)[TJ] = wr[u & 1];
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(bf16x8, wc[j]), __builtin_bit_cast(bf16x8, xc[i]),
                        acc[i][j], 0, 0, 0);
        }
    }
    if constexpr (STAGED && EPI == kDenseStore) {
        if (a.vec_out == 2) {
            barrier_no_fence();  // every wave is done with the stage buffers
            dense_store_staged<T, TI, TJ>(a, acc, smem + wave * WM * staged_pitch<T, WN>(), p0 + wm * WM,
                                          n0 + wn * WN, h, r, lane);
            return;
        }
    }
    dense_epilogue<T, TI, TJ, EPI>(a, acc, p0 + wm * WM, n0 + wn * WN, h, r);
}

// ---- fp32 products on the bf16 matrix cores --------------------------------
// Each fp32 operand is split into three bf16 terms and a product takes six of
// their products (split3.h).  Six v_mfma_f32_32x32x16_bf16 cost 192 matrix-core cycles where the eight
// v_mfma_f32_32x32x2_f32 of the same 16 K steps cost 512.  Against 64-bit
// products of N(0, 1) operands the results are closer than that instruction's:
// relative error (2-norm) 3.4e-7 against 4.0e-7 at K = 1024, 7.1e-7 against
// 8.1e-7 at 4096, 8.1e-8 against 1.05e-7 at 64.
//
// What bounds it: the vector instructions that split the operands (12 per pair
// of values) beside the matrix cores, so a split is shared by as large a tile
// as registers and a balanced grid allow.  206,980 x 1024 -> 256: 627 us
// against 873 on fp32 MFMA tiles (173 against 124 TFLOP/s); 4,736 x 1024 ->
// 4096: 224 against 315; 1,000 x 4096 -> 1024: 105 against 155.  Tiles of 256 x
// 256 or 256 x 128 (8 or 16 waves, one workgroup per CU) ran slower: 683-1,173
// us on the first shape.
// One tile of BM x BN, NWM x NWN waves.  Per 32-element K chunk every thread
// splits its share of the X and W rows (loaded into registers while the chunk
// before is multiplied) and writes the planes to LDS as [plane][8-element
// piece][row] pieces of 16 bytes (piece columns 64 bytes apart modulo the
// banks, so that the 4 pieces of a row that neighbouring lanes write do not
// conflict; fragment reads cover 256 contiguous bytes per 16 lanes).
template <int BM, int BN, int NWM, int NWN, int WPE, int EPI>
__global__ void __launch_bounds__(NWM * NWN * 64) __attribute__((amdgpu_waves_per_eu(WPE)))
dense_split_kernel(DenseArgs a) {
    constexpr int NT = NWM * NWN * 64, RS = NT / 8;  // rows apart a thread's pieces are
    constexpr int WM = BM / NWM, WN = BN / NWN, TI = WM / 32, TJ = WN / 32;
    constexpr int kColX = BM * 16 + 64, kColW = BN * 16 + 64;  // bytes per piece column
    constexpr int kPlaneX = 4 * kColX, kPlaneW = 4 * kColW;
    constexpr int XI = BM / RS, WI = BN / RS;  // pieces per thread and chunk
    extern __shared__ __align__(16) char smem[];
    char * sx = smem;
    char * sw = smem + 3 * kPlaneX;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / NWN, wn = wave % NWN;
    const int h = lane >> 5, r = lane & 31;
    const int tiles_n = (a.n + BN - 1) / BN;
    const int tiles_m = static_cast<int>((a.m + BM - 1) / BM);
    int tm, tn;
    tile_of(remap_xcd(blockIdx.x, gridDim.x), tiles_m, tiles_n, a.group_m, tm, tn);
    const int64_t p0 = static_cast<int64_t>(tm) * BM;
    const int n0 = tn * BN;
    const float * x = static_cast<const float *>(a.x);
    const float * w = static_cast<const float *>(a.w);

    // This thread's 16-byte pieces of the 128-byte chunk rows: piece `piece`,
    // rows row + RS i (clamped; outputs past the end are not stored).
    const int piece = tid & 7, row = tid >> 3;
    const char * xb = reinterpret_cast<const char *>(x + p0 * a.k);
    const char * wb = reinterpret_cast<const char *>(w + static_cast<int64_t>(n0) * a.k);
    const int64_t last_x = a.m - 1 - p0;
    const int last_w = a.n - 1 - n0;
    uint32_t x_off[XI], w_off[WI];  // bytes
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int m = row + RS * i;
        x_off[i] = static_cast<uint32_t>(((m < last_x ? m : last_x) * a.k + piece * 4) * 4);
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int n = row + RS * i;
        w_off[i] = static_cast<uint32_t>((static_cast<int64_t>(n < last_w ? n : last_w) * a.k + piece * 4) * 4);
    }
    // K chunks of this workgroup: all, or its split's share of them.
    const int all_chunks = (a.k + 31) / 32;
    int chunk0 = 0, chunks = all_chunks;
    if constexpr (EPI == kDensePartial) {
        chunk0 = static_cast<int>(blockIdx.y) * all_chunks / a.splits;
        chunks = (static_cast<int>(blockIdx.y) + 1) * all_chunks / a.splits - chunk0;
        a.residual += static_cast<int64_t>(blockIdx.y) * a.m * a.n;
    }
    float4 vx[XI], vw[WI];
    auto load = [&](int s) __attribute__((always_inline)) {
        const char * xs = xb + static_cast<int64_t>(s) * 128;
        const char * wsb = wb + static_cast<int64_t>(s) * 128;
        if (s * 32 + 32 <= a.k) {
#pragma unroll
            for (int i = 0; i < XI; ++i) vx[i] = *reinterpret_cast<const float4 *>(xs + x_off[i]);
#pragma unroll
            for (int i = 0; i < WI; ++i) vw[i] = *reinterpret_cast<const float4 *>(wsb + w_off[i]);
        } else {
            const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const bool in = s * 32 + piece * 4 < a.k;
#pragma unroll
            for (int i = 0; i < XI; ++i) {
                vx[i] = zero;
                if (in) vx[i] = *reinterpret_cast<const float4 *>(xs + x_off[i]);
            }
#pragma unroll
            for (int i = 0; i < WI; ++i) {
                vw[i] = zero;
                if (in) vw[i] = *reinterpret_cast<const float4 *>(wsb + w_off[i]);
            }
        }
    };

    f32x16 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    float hi = 0.0f;
    load(chunk0);
    for (int s = 0; s < chunks; ++s) {
        barrier_no_fence();  // every wave has read the previous chunk
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            uint2 t[3];
            split4(vx[i], t, hi);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<uint2 *>(sx + q * kPlaneX + (piece >> 1) * kColX + (row + RS * i) * 16 + (piece & 1) * 8) = t[q];
        }
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            uint2 t[3];
            split4(vw[i], t, hi);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<uint2 *>(sw + q * kPlaneW + (piece >> 1) * kColW + (row + RS * i) * 16 + (piece & 1) * 8) = t[q];
        }
        if (s + 1 < chunks) load(chunk0 + s + 1);
        barrier_no_fence();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            bf16x8 xf[3][TI];
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int i = 0; i < TI; ++i)
                    xf[q][i] = *reinterpret_cast<const bf16x8 *>(
                        sx + q * kPlaneX + (2 * u + h) * kColX + (wm * WM + i * 32 + r) * 16);
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                bf16x8 wf[3];
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    wf[q] = *reinterpret_cast<const bf16x8 *>(
                        sw + q * kPlaneW + (2 * u + h) * kColW + (wn * WN + j * 32 + r) * 16);
#pragma unroll
                for (int t = 0; t < 6; ++t)
#pragma unroll
                    for (int i = 0; i < TI; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[kSplitTermB[t]], xf[kSplitTermA[t]][i],
                                                                            acc[i][j], 0, 0, 0);
            }
        }
    }
    // A split's share of K has the whole K's bound: the rule then is one of rows and
    // channels, whatever the split.
    bool odd = hi > kSplitHigh;
    const float low = split_low(kSplitHigh, a.k);
    float sum[TI][TJ][16];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                sum[i][j][v] = acc[i][j][v];
                asm("" : "+v"(sum[i][j][v]));  // scalars from here on: vectors would be copied whole, and spill
                odd |= split_sum_odd(sum[i][j][v], low);
            }
    if (__builtin_expect(__syncthreads_or(odd), 0)) {
        hi = split_block_max(hi, reinterpret_cast<uint32_t *>(smem));
        const float tile_low = split_low(hi, a.k);
        bool again = hi > kSplitHigh, zero = false;
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    zero |= sum[i][j][v] == 0.0f;
                    again |= sum[i][j][v] != 0.0f && split_sum_odd(sum[i][j][v], tile_low);
                }
        const int k_end = min(a.k, (chunk0 + chunks) * 32);  // a multiple of 4, as chunk0 * 32 is
        if (__syncthreads_or(zero)) {
            // Zeros of zero rows, or of zero channels, are what they should be, and of the
            // others (of sums that cancel, about one output in 2^28) those without small operands.
            // So only the rows and channels that hold a zero are looked through.
            uint32_t * flags = reinterpret_cast<uint32_t *>(smem);  // BM rows, then BN channels
            for (int i = tid; i < (BM + BN) / 32; i += NT) flags[i] = 0u;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j) {
                    bool any = false;
                    uint32_t channels = 0;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const bool z = sum[i][j][v] == 0.0f;
                        any |= z;
                        const uint64_t lanes = __ballot(z);
                        channels |= (static_cast<uint32_t>(lanes) ? 1u : 0u) << (8 * (v >> 2) + (v & 3));
                        channels |= (lanes >> 32 ? 1u : 0u) << (8 * (v >> 2) + 4 + (v & 3));
                    }
                    const uint64_t rows = __ballot(any);
                    if (lane == 0) {
                        atomicOr(flags + (wm * WM) / 32 + i, static_cast<uint32_t>(rows | rows >> 32));
                        atomicOr(flags + (BM + wn * WN) / 32 + j, channels);
                    }
                }
            __syncthreads();
            int in_x = 0, in_w = 0;
            for (int i = 0; i < BM / 32; ++i) in_x += __popc(flags[i]);
            for (int i = BM / 32; i < (BM + BN) / 32; ++i) in_w += __popc(flags[i]);
            // The marked lines of X or W: whether one is not all zero, whether one holds a
            // small operand.  Few lines: each over all threads; many: 256 inputs of all lines
            // at a time, and with `first` only up to the first operand that is not zero.
            auto look = [&](bool of_x, bool few, bool first, bool & nonzero, bool & small) {
                const int base = of_x ? 0 : BM, count = of_x ? BM : BN;
                auto line = [&](int i) -> const float * {
                    return of_x ? x + (p0 + (i < last_x ? i : last_x)) * a.k
                                : w + static_cast<int64_t>(n0 + (i < last_w ? i : last_w)) * a.k;
                };
                auto marked = [&](int i) { return (flags[(base + i) / 32] >> (i & 31) & 1u) != 0; };
                if (few) {
                    for (int i0 = 0; i0 < count; i0 += 32)
                        for (uint32_t left = flags[(base + i0) / 32]; left != 0; left &= left - 1) {
                            const float * p = line(i0 + __ffs(left) - 1);
                            for (int k = chunk0 * 32 + tid * 4; k < k_end; k += NT * 4) {
                                const float4 f = *reinterpret_cast<const float4 *>(p + k);
                                nonzero |= max_abs(f) != 0.0f;
                                small |= split_small(f);
                            }
                        }
                    return;
                }
                for (int k0 = chunk0 * 32; k0 < k_end; k0 += 256) {
                    for (int i = row; i < count; i += RS) {
                        if (!marked(i)) continue;
                        const float * p = line(i);
#pragma unroll 4
                        for (int k = k0 + piece * 4; k < min(k0 + 256, k_end); k += 32) {
                            const float4 f = *reinterpret_cast<const float4 *>(p + k);
                            nonzero |= max_abs(f) != 0.0f;
                            small |= split_small(f);
                        }
                    }
                    if (first && __syncthreads_or(nonzero)) return;
                }
            };
            const bool few_x = in_x <= 16, few_w = in_w <= 16;
            bool clean = false, small = false;
#pragma unroll 1
            for (int pass = 0; pass < 2 && !clean; ++pass) {
                const bool of_x = (in_x <= in_w) == (pass == 0);
                bool nonzero = false, found = false;
                look(of_x, of_x ? few_x : few_w, true, nonzero, found);
                clean = !__syncthreads_or(nonzero);
                small |= found;
            }
            if (!clean) {
                bool unused = false;
                if (!few_x) look(true, false, false, unused, small);
                if (!few_w) look(false, false, false, unused, small);
                again |= small;
            }
        }
        if (__syncthreads_or(again)) {
            // One 32 x 32 block at a time, its sums picked out and put back by number:
            // with the blocks' loops written out one after the other registers spilled.
#pragma unroll 1
            for (int b = 0; b < TI * TJ; ++b) {
                const int64_t m = p0 + wm * WM + b / TJ * 32 + r;
                const int n = n0 + wn * WN + b % TJ * 32 + r;
                const float * xr = x + (m < a.m ? m : a.m - 1) * a.k;
                const float * wr = w + static_cast<int64_t>(n < a.n ? n : a.n - 1) * a.k;
                f32x16 second = {};
                float hi_x = 0.0f, hi_w = 0.0f;
                bool small_x = false, small_w = false;
                for (int k = chunk0 * 32 + 4 * h; k - 4 * h < k_end; k += 8) {
                    float4 fx = make_float4(0.0f, 0.0f, 0.0f, 0.0f), fw = fx;
                    if (k < k_end) {
                        fx = *reinterpret_cast<const float4 *>(xr + k);
                        fw = *reinterpret_cast<const float4 *>(wr + k);
                    }
                    hi_x = fmaxf(hi_x, max_abs(fx));
                    hi_w = fmaxf(hi_w, max_abs(fw));
                    small_x |= split_small(fx);
                    small_w |= split_small(fw);
                    second = __builtin_amdgcn_mfma_f32_32x32x2f32(fw.x, fx.x, second, 0, 0, 0);
                    second = __builtin_amdgcn_mfma_f32_32x32x2f32(fw.y, fx.y, second, 0, 0, 0);
                    second = __builtin_amdgcn_mfma_f32_32x32x2f32(fw.z, fx.z, second, 0, 0, 0);
                    second = __builtin_amdgcn_mfma_f32_32x32x2f32(fw.w, fx.w, second, 0, 0, 0);
                }
                float block[16];
#pragma unroll
                for (int v = 0; v < 16; ++v) block[v] = sum[0][0][v];
#pragma unroll
                for (int q = 1; q < TI * TJ; ++q)
#pragma unroll
                    for (int v = 0; v < 16; ++v) block[v] = q == b ? sum[q / TJ][q % TJ][v] : block[v];
                split_select(block, second, hi_w, hi_x, small_w, small_x, a.k, h);
#pragma unroll
                for (int q = 0; q < TI * TJ; ++q)
#pragma unroll
                    for (int v = 0; v < 16; ++v) sum[q / TJ][q % TJ][v] = q == b ? block[v] : sum[q / TJ][q % TJ][v];
            }
        }
        __syncthreads();  // the words in smem have been read
    }
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = sum[i][j][v];
    if constexpr (EPI == kDenseStore) {
        if (a.vec_out == 2) {
            // 32 rows of each wave's block at a time through the idle planes
            barrier_no_fence();
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                f32x16 part[1][TJ];
#pragma unroll
                for (int j = 0; j < TJ; ++j) part[0][j] = acc[i][j];
                dense_store_staged<float, 1, TJ>(a, part, smem + wave * 32 * staged_pitch<float, WN>(),
                                                 p0 + wm * WM + i * 32, n0 + wn * WN, h, r, lane);
            }
            return;
        }
    }
    dense_epilogue<float, TI, TJ, EPI>(a, acc, p0 + wm * WM, n0 + wn * WN, h, r);
}

template <int BM, int BN, int NWM, int NWN, int WPE, int EPI>
int launch_dense_split(const DenseArgs & a, hipStream_t stream) {
    constexpr int kPlanes = 3 * 4 * ((BM + BN) * 16 + 128);
    constexpr int kStaged = EPI == kDenseStore ? NWM * NWN * 32 * staged_pitch<float, BN / NWN>() : 0;
    constexpr int smem = kPlanes > kStaged ? kPlanes : kStaged;
    auto kernel = &dense_split_kernel<BM, BN, NWM, NWN, WPE, EPI>;
    if constexpr (smem > 64 * 1024) {
        static bool configured = false;
        if (!configured) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, smem);
            if (e != hipSuccess) return check_hip(e, "hipFuncSetAttribute(dense_split)");
            configured = true;
        }
    }
    const int64_t blocks = ((a.m + BM - 1) / BM) * ((a.n + BN - 1) / BN);
    if (blocks > INT32_MAX) return fail(PXS_ERR_ARG, "dense GEMM grid too large");
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks), EPI == kDensePartial ? a.splits : 1),
                       dim3(NWM * NWN * 64), smem, stream, a);
    return check_launch("dense GEMM (fp32 split)");
}

template <typename T, int BM, int BN, int NW, int WAVES_M, int NSTAGE, int KB, int EPI,
          bool SPREAD, bool STAGED, typename... GROUP>
int launch_dense(const DenseArgs & a, hipStream_t stream, int count = 1, const GROUP &... group) {
    constexpr int kStage = (BM + BN) * KB;
    constexpr int kChunk = KB / static_cast<int>(sizeof(T));
    constexpr int WN = BN / (NW / WAVES_M);
    constexpr int kStagedBytes = STAGED && EPI == kDenseStore ? NW * (BM / WAVES_M) * staged_pitch<T, WN>() : 0;
    constexpr int kMaxSmem = NSTAGE * kStage > kStagedBytes ? NSTAGE * kStage : kStagedBytes;
    static_assert(kMaxSmem <= 160 * 1024, "LDS");
    auto kernel = &dense_gemm_kernel<T, BM, BN, NW, WAVES_M, NSTAGE, KB, EPI, SPREAD, STAGED, GROUP...>;
    static bool configured = false;
    if (!configured) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, kMaxSmem);
        if (e != hipSuccess) return check_hip(e, "hipFuncSetAttribute(dense_gemm)");
        configured = true;
    }
    const int stages = (a.k + kChunk - 1) / kChunk;
    int smem = (stages < NSTAGE ? stages : NSTAGE) * kStage;
    if (a.vec_out == 2 && smem < kStagedBytes) smem = kStagedBytes;
    const int64_t blocks = ((a.m + BM - 1) / BM) * ((a.n + BN - 1) / BN);
    if (blocks > INT32_MAX) return fail(PXS_ERR_ARG, "dense GEMM grid too large");
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks), EPI == kDensePartial ? a.splits : count),
                       dim3(NW * 64), smem, stream, a, group...);
    return check_launch("dense GEMM");
}

// fp32 linears of 1 to kFewRows rows (a flow's timestep embedding and its
// modulation): one wave per output channel reads its weight row once, 16 bytes
// per lane, and a tile of 64 rows would have run nearly empty: 1 x 1024 -> 6144
// (25 MB of weights) 39 us on 64 x 64 tiles.  blockIdx.y: each kFewRows rows.
constexpr int kFewRows = 4;
__global__ void __launch_bounds__(256)
few_rows_f32_kernel(DenseArgs a) {
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (n >= a.n) return;
    const float * w = static_cast<const float *>(a.w) + static_cast<int64_t>(n) * a.k;
    const int m0 = blockIdx.y * kFewRows, rows = min(static_cast<int>(a.m) - m0, kFewRows);
    const float * x = static_cast<const float *>(a.x) + static_cast<int64_t>(m0) * a.k;
    float sum[kFewRows] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int k = lane * 4; k < a.k; k += 256) {
        const float4 f = *reinterpret_cast<const float4 *>(w + k);
#pragma unroll
        for (int m = 0; m < kFewRows; ++m) {
            if (m >= rows) break;
            const float4 v = *reinterpret_cast<const float4 *>(x + static_cast<int64_t>(m) * a.k + k);
            sum[m] = fmaf(f.x, v.x, sum[m]);
            sum[m] = fmaf(f.y, v.y, sum[m]);
            sum[m] = fmaf(f.z, v.z, sum[m]);
            sum[m] = fmaf(f.w, v.w, sum[m]);
        }
    }
#pragma unroll
    for (int m = 0; m < kFewRows; ++m) {
        if (m >= rows) break;
        float v = sum[m];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
        v += a.bias ? a.bias[n] : 0.0f;
        if (a.act == PXS_ACT_GELU_TANH) v = gelu_tanh_f(v);
        else if (a.act == PXS_ACT_SILU) v = silu_f(v);
        if (lane == 0) static_cast<float *>(a.y)[static_cast<int64_t>(m0 + m) * a.n + n] = v;
    }
}

// Tile shape by the estimated time of the whole grid: rounds of tiles over
// the 256 CUs (workgroups resident per CU in parallel) times the time of one
// round, from each shape's measured rate (256 x 256 tiles about 1000 TFLOP/s,
// 128 x 128 about 880, 128 x 64 about 700).  256 x 256 tiles go down
// 8-row-tile groups, the others down groups of 16 when a row holds at most 4
// column tiles, else 8.
template <int EPI>
int dispatch_bf16(DenseArgs a, hipStream_t s) {
    auto rounds = [&](int bm, int bn, int per_cu) {
        const int64_t tiles = ((a.m + bm - 1) / bm) * ((a.n + bn - 1) / bn);
        return static_cast<double>((tiles + 256 * per_cu - 1) / (256 * per_cu));
    };
    const double t_a = rounds(256, 256, 1) * 256.0 * 256 / 1000.0;
    const double t_b = rounds(128, 128, 2) * 2.0 * 128 * 128 / 880.0;
    const double t_c = rounds(128, 64, 3) * 3.0 * 128 * 64 / 700.0;
    if (a.n > 128 && t_a <= t_b) {
        a.group_m = 8;
        return launch_dense<uint16_t, 256, 256, 16, 4, 2, 128, EPI, true, true>(a, s);
    }
    // At most one 128 x 64 tile per CU: nothing else hides a workgroup's waits, so
    // 8 waves of 32 x 32 and three stages (1,000 x 1024 -> 1024: 10.1 against 12.4
    // us, 4096 -> 1024: 29 against 38 us; 300 x 1024 -> 4096: 10.2 against 12.5 us).
    if (((a.m + 127) / 128) * ((a.n + 63) / 64) <= 256) {
        a.group_m = 8;
        return launch_dense<uint16_t, 128, 64, 8, 4, 3, 128, EPI, false, true>(a, s);
    }
    if (a.n <= 64 || t_c < t_b) {
        a.group_m = (a.n + 63) / 64 <= 4 ? 16 : 8;
        return launch_dense<uint16_t, 128, 64, 4, 2, 2, 128, EPI, false, true>(a, s);
    }
    a.group_m = (a.n + 127) / 128 <= 4 ? 16 : 8;
    return launch_dense<uint16_t, 128, 128, 8, 2, 2, 128, EPI, false, true>(a, s);
}

// fp32: the tile with the least estimated time, in us per 1024 of K: what a
// lone workgroup takes, or the workgroups a CU gets times what each adds
// (measured on 1,000 to 206,980 rows).  A tie goes to the larger tile.
template <int EPI>
int dispatch_f32(DenseArgs a, hipStream_t s) {
    auto time = [&](int bm, int bn, double alone, double each) {
        const int64_t tiles = ((a.m + bm - 1) / bm) * ((a.n + bn - 1) / bn);
        return std::max(alone, static_cast<double>((tiles + 255) / 256) * each);
    };
    const double t_a = time(128, 128, 64.0, 48.0), t_b = time(128, 64, 44.0, 28.0);
    const double t_c = time(64, 64, 31.0, 16.0);
    a.group_m = 8;
    if (a.n > 64 && t_a <= t_b && t_a <= t_c) return launch_dense_split<128, 128, 2, 2, 3, EPI>(a, s);
    if (t_b <= t_c) return launch_dense_split<128, 64, 2, 2, 3, EPI>(a, s);
    return launch_dense_split<64, 64, 2, 2, 4, EPI>(a, s);
}

bool aligned_to(const void * p, uintptr_t bytes) { return (reinterpret_cast<uintptr_t>(p) % bytes) == 0; }

// Common checks; false when the kernel does not take the shape (rows of X or
// W not whole 16-byte pieces, or operands not 16-byte aligned).
bool dense_takes(int dtype, const void * x, int cin, const void * w) {
    const int vec = dtype == PXS_BF16 ? 8 : 4;
    return (dtype == PXS_BF16 || dtype == PXS_F32) && cin % vec == 0 && aligned_to(x, 16) &&
           aligned_to(w, 16);
}

template <int EPI>
int run_dense(int dtype, const DenseArgs & a, hipStream_t s) {
    return dtype == PXS_BF16 ? dispatch_bf16<EPI>(a, s) : dispatch_f32<EPI>(a, s);
}

} // namespace

int dense_linear(int dtype, const void * x, int64_t rows, int cin, const void * w,
                 const float * bias, int cout, int act, void * y, int64_t plan_rows, hipStream_t s,
                 bool * done) {
    *done = false;
    if (!dense_takes(dtype, x, cin, w)) return PXS_OK;
    DenseArgs a{};
    a.x = x; a.w = w; a.bias = bias; a.m = rows; a.k = cin; a.n = cout; a.y = y; a.act = act;
    a.vec_out = cout % 4 == 0 && aligned_to(y, dtype == PXS_BF16 ? 8 : 16) &&
                (!bias || aligned_to(bias, 16));
    // Whole 16-byte pieces of output rows: the store goes through LDS.
    if (a.vec_out && cout % (dtype == PXS_BF16 ? 8 : 4) == 0 && aligned_to(y, 16)) a.vec_out = 2;
    *done = true;
    if (dtype == PXS_F32 && rows > 0 && plan_rows <= kFewRows) {
        hipLaunchKernelGGL(few_rows_f32_kernel, dim3(grid_for(cout, 4), grid_for(rows, kFewRows)), dim3(256), 0,
                           s, a);
        return check_launch("linear of few rows");
    }
    return run_dense<kDenseStore>(dtype, a, s);
}

int dense_linear_residual(int dtype, const void * x, int64_t rows, int cin, const void * w,
                          const float * bias, int cout, float * residual, hipStream_t s,
                          bool * done) {
    *done = false;
    if (!dense_takes(dtype, x, cin, w)) return PXS_OK;
    DenseArgs a{};
    a.x = x; a.w = w; a.bias = bias; a.m = rows; a.k = cin; a.n = cout; a.residual = residual;
    a.vec_out = cout % 4 == 0 && aligned_to(residual, 16) && (!bias || aligned_to(bias, 16));
    *done = true;
    return run_dense<kDenseAddResidual>(dtype, a, s);
}

int dense_linear_gate(int dtype, const void * x, int64_t rows, int cin, const void * w,
                      const float * bias, int cout, const int32_t * coords,
                      const float * block_mod, const float * time_mod, int gate_offset,
                      float * residual, hipStream_t s, bool * done) {
    *done = false;
    if (!dense_takes(dtype, x, cin, w)) return PXS_OK;
    DenseArgs a{};
    a.x = x; a.w = w; a.bias = bias; a.m = rows; a.k = cin; a.n = cout; a.residual = residual;
    a.coords = coords; a.block_mod = block_mod; a.time_mod = time_mod; a.gate_offset = gate_offset;
    a.vec_out = cout % 4 == 0 && gate_offset % 4 == 0 && aligned_to(residual, 16) &&
                (!bias || aligned_to(bias, 16)) && aligned_to(block_mod, 16) &&
                aligned_to(time_mod, 16);
    *done = true;
    return run_dense<kDenseGate>(dtype, a, s);
}

// bf16 linears of one input with up to kDenseGroup weights [cout, cin] and
// biases, in one launch: y [count, rows, cout].
bool dense_group_takes(int cin, int cout) { return cin % 8 == 0 && cout % 8 == 0 && cout > 128; }

int dense_linear_group(const void * x, int64_t rows, int cin, const void * const * w,
                       const float * const * bias, int count, int cout, void * y, hipStream_t s) {
    PXS_CHECK(count > 0 && count <= kDenseGroup, PXS_ERR_ARG, "dense linear group: bad count");
    DenseGroup g{};
    for (int i = 0; i < count; ++i) {
        g.w[i] = w[i];
        g.bias[i] = bias[i];
    }
    DenseArgs a{};
    a.x = x; a.m = rows; a.k = cin; a.n = cout; a.y = y;
    a.vec_out = 2;
    a.group_m = 8;
    return launch_dense<uint16_t, 256, 256, 16, 4, 2, 128, kDenseStore, true, true, DenseGroup>(a, s, count, g);
}

// Few rows leave most CUs without a 128 x 128 tile, and smaller tiles move
// more operand bytes per product through each CU (about 40 GB/s, the bound
// here: 1,000 x 4096 -> 1024 in bf16 takes 38 us on 128 x 64 tiles and 28 us on
// 64 x 64 tiles, with two stages in flight or six).  K is then split so that
// the tiles come near to one per CU.
// Six blocks of width 1024 with their three residual linears in one pass
// against 2, 3, 4, 5 splits: 248 rows 1,775 us against 1,628, 1,596, 1,586, 1,590;
// 1,288 rows 1,632 against 1,500, 1,515, 1,508, 1,539; 2,600 rows (168 tiles) 2,118
// against 2,037, 2,077, 2,202, 2,229; 4,064 rows (256 tiles) 2,503 against 2,522,
// 2,698, 2,736, 2,863.
// So up to 170 tiles, by the call alone.  A guided step runs the rows of a call twice
// with the splits of one branch (Branches) where those of the doubled batch would
// suit it better past 104 tiles: two guided steps of four blocks of width 1024, 1,600
// rows (104 tiles) 2,870 us against 2,956 in one pass, 2,600 rows (168) 4,160 against
// 3,956.  A line at 104 would cost one forward alone as much (2,100 rows 1,255 us
// against 1,171).
constexpr int64_t kSplitTiles = 170;
int dense_splits(int dtype, int64_t rows, int cin, int cout) {
    const int vec = dtype == PXS_BF16 ? 8 : 4, chunk = 8 * vec;
    if (rows <= 0 || cin % vec != 0 || cout % 4 != 0 || cout <= 64) return 0;
    const int64_t tiles = ((rows + 127) / 128) * ((cout + 127) / 128);
    if (tiles > kSplitTiles) return 0;
    const int64_t most = std::min<int64_t>(4, cin / (4 * chunk));  // 4 stages of K each
    const int64_t splits = std::min(most, std::max<int64_t>(2, 256 / tiles));
    return splits >= 2 ? static_cast<int>(splits) : 0;
}

int64_t dense_split_rows(int dtype, int64_t rows, int cin, int cout) {
    int64_t most = 0;
    if (cout <= 0) return 0;  // (a size query takes any configuration)
    const int64_t row_tiles = std::min((rows + 127) / 128, kSplitTiles / ((cout + 127) / 128));
    for (int64_t t = 1; t <= row_tiles; ++t) {  // the splits depend on the row tiles only
        const int64_t r = std::min(rows, 128 * t);
        most = std::max(most, dense_splits(dtype, r, cin, cout) * r);
    }
    return most;
}

int dense_partial(int dtype, const void * x, int64_t rows, int cin, const void * w, int cout,
                  int splits, float * partial, hipStream_t s) {
    DenseArgs a{};
    a.x = x; a.w = w; a.m = rows; a.k = cin; a.n = cout; a.residual = partial; a.splits = splits;
    a.vec_out = 1;
    a.group_m = 8;
    return dtype == PXS_BF16
               ? launch_dense<uint16_t, 128, 128, 8, 2, 2, 128, kDensePartial, false, false>(a, s)
               : launch_dense_split<128, 128, 2, 2, 3, kDensePartial>(a, s);
}

} // namespace pxs
