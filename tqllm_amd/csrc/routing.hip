// Router logits, softmax + top-k, and the stable token-to-expert dispatch.
#include <atomic>
#include <mutex>

#include "act_image.cuh"
#include "lds_dma.cuh"
#include "common.cuh"
#include "grouped_plan.cuh"
#include "routing_api.cuh"
#include "row_quant.cuh"
#include "topk_select.cuh"

namespace tqmoe {
namespace {

// ----------------------------------------------------------------------------------------------------- router
// One wave per router row, TOK tokens per pass; each lane owns 8-element chunks lane, lane + 64, ... of the row.
// Sums in fp32; the order (chunks ascending per lane, then a butterfly over lanes) differs from a column-order host
// sum by ordinary fp32 rounding only.
constexpr int kRouterTok = 4;       // tokens per pass of a wave: the router row is read once for them
constexpr int kRouterTokFew = 1;    // decode-sized batches: a wave per (row, token), the latency of a wave's chain is what counts
template <int WT, int XT, int TOK>
__global__ __launch_bounds__(256) void router_k(const void * __restrict__ w, const void * __restrict__ shared,
                                                const void * __restrict__ x, float * __restrict__ logits, int h, int e, int n, RouterSide side) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if ((side.image || side.zero) && blockIdx.x == gridDim.x - 1) {   // a further block per pass for what stands beside the routing
        if (blockIdx.y == 0)
            for (int i = threadIdx.x; i < side.zero_n; i += 256) side.zero[i] = 0;
        if constexpr (TOK == 1) {
            if (side.image && wave == 0) quantise_row_wave<XT>(x, blockIdx.y, h, side.image + int64_t(blockIdx.y) * (h / 32) * kImageSubBytes, lane);
        }
        return;
    }
    const int row = blockIdx.x * 4 + wave;  // 0..e (e = the shared gate)
    const int t0 = blockIdx.y * TOK;
    if (row > e) return;                     // whole waves leave together: reductions below see full waves
    const bool has_row = row < e || shared != nullptr;
    const void * wr = row < e ? w : shared;
    const int64_t wbase = row < e ? int64_t(row) * h : 0;
    float acc[TOK];
#pragma unroll
    for (int i = 0; i < TOK; ++i) acc[i] = 0.f;
    if (has_row) {
        // four 512-column steps of loads at a time (one trip to memory for them instead of four), the sums in column order
        // as before; then what is left of the row step by step
        int c = lane * 8;
        if constexpr (TOK > 1) {   // two steps of loads at a time for the four tokens of a pass
            for (; c + 512 < h; c += 2 * 512) {
                float wv[2][8], xv[TOK][2][8];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    load8<WT>(wr, wbase + c + 512 * q, wv[q]);
#pragma unroll
                    for (int i = 0; i < TOK; ++i) load8<XT>(x, int64_t(min(t0 + i, n - 1)) * h + c + 512 * q, xv[i][q]);
                }
#pragma unroll
                for (int i = 0; i < TOK; ++i)
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int j = 0; j < 8; ++j) acc[i] = fmaf(wv[q][j], xv[i][q][j], acc[i]);
            }
        }
        if constexpr (TOK == 1) {
            for (; c + 3 * 512 < h; c += 4 * 512) {
                float wv[4][8], xv[4][8];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    load8<WT>(wr, wbase + c + 512 * q, wv[q]);
                    load8<XT>(x, int64_t(t0) * h + c + 512 * q, xv[q]);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[0] = fmaf(wv[q][j], xv[q][j], acc[0]);
            }
        }
        for (; c < h; c += 512) {
            float wv[8];
            load8<WT>(wr, wbase + c, wv);
#pragma unroll
            for (int i = 0; i < TOK; ++i) {
                if (t0 + i < n) {
                    float xv[8];
                    load8<XT>(x, int64_t(t0 + i) * h + c, xv);
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[i] = fmaf(wv[j], xv[j], acc[i]);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < TOK; ++i) {
        const float s = group_sum<64>(acc[i]);
        if (lane == 0 && t0 + i < n) logits[int64_t(t0 + i) * (e + 1) + row] = s;
    }
}

template <int WT> int32_t launch_router_x(uint32_t xtype, const void * w, const void * sg, const void * x, float * logits,
                                          int h, int e, int n, const RouterSide & side, hipStream_t s) {
    const bool wide = n <= kRouterFew || side.image;   // the wide grid of one-token passes (which write the activation images)
    const int tok = wide ? kRouterTokFew : kRouterTok;
    const dim3 grid(unsigned((e + 1 + 3) / 4 + (side.image || side.zero ? 1 : 0)), unsigned((n + tok - 1) / tok));
    switch (xtype) {
        case TQMOE_F32:
            if (wide) router_k<WT, TQMOE_F32, kRouterTokFew><<<grid, 256, 0, s>>>(w, sg, x, logits, h, e, n, side);
            else router_k<WT, TQMOE_F32, kRouterTok><<<grid, 256, 0, s>>>(w, sg, x, logits, h, e, n, side);
            return 0;
        case TQMOE_F16:
            if (wide) router_k<WT, TQMOE_F16, kRouterTokFew><<<grid, 256, 0, s>>>(w, sg, x, logits, h, e, n, side);
            else router_k<WT, TQMOE_F16, kRouterTok><<<grid, 256, 0, s>>>(w, sg, x, logits, h, e, n, side);
            return 0;
        case TQMOE_BF16:
            if (wide) router_k<WT, TQMOE_BF16, kRouterTokFew><<<grid, 256, 0, s>>>(w, sg, x, logits, h, e, n, side);
            else router_k<WT, TQMOE_BF16, kRouterTok><<<grid, 256, 0, s>>>(w, sg, x, logits, h, e, n, side);
            return 0;
    }
    return -1;
}

// Router logits of more tokens, bf16 rows on both sides or fp32 rows on both sides: a GEMM on the matrix pipe. bf16 x bf16
// products are exact in fp32, the fp32 instruction multiplies and adds in fp32, and both accumulate in fp32, so the result
// differs from the scalar kernel's only by the order of the sum.
// A block of eight waves takes 16 TA tokens x 64 router rows; every wave computes the whole tile over an eighth of the
// columns, operands straight from memory (16 bytes a lane, 64 of a row together), a chunk of steps ahead of the matrix
// instructions, and the eight partial tiles are added through LDS in a fixed order. No stage is waited for by the whole block:
// a launch is one trip to memory and the bandwidth of the L2, where stages of 256 columns through LDS were a chain of eight
// trips (512 experts, 2048 columns: 21 us for 333 tokens, 32 for 4096). TA is the largest tile that still gives every
// compute unit a block; one of 16 tokens goes through LDS after all, each wave's operands by themselves (router_gemm_dma_k), and is
// left here for operands that are not aligned to 16 bytes. A token's sums do not depend on any of this, nor on the batch.
// The last row of blocks takes the shared expert's gate row (or stores its zeros): a wave a token.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
// Tokens x router rows from which a router and input of one type take the GEMM. Drawn for tiles straight from memory, which bf16 rows that are not
// aligned have (us, wave per row / GEMM, 40000: 1024 columns 6.9 / 7.3, 2048 9.6 / 11.7, 4096 17.5 / 20.5). Aligned rows, whose small tiles go
// through LDS, cross at fewer (31 to 1000 experts; us at 33000): bf16 with 1024 columns at 26000 (5.7 / 5.0), with 2048 at 22000 (8.0 / 6.1), with 4096
// at 16000 (13.1 / 8.2); fp32 with 1024 at 45000, with 2048 at 33000 to 41000 (13.5 / 15.3 to 18.3 / 15.5), with 4096 at 24000 to 33000 (34 / 27).
// The line stays for them as well: eight slices of a row on the matrix pipe are further from 64 bits than a wave's sums (root of the mean square over
// the logits', wave per row / GEMM: bf16 2048 columns 7.5e-8 / 9.8e-8, 4096 8.4e-8 / 1.33e-7; fp32 1.23e-7 / 2.89e-7, 1.59e-7 / 4.07e-7), and no
// batch is to get coarser logits than it had.
template <bool F32> constexpr int kRouterGemmMin = F32 ? 56000 : 45000;
constexpr int kRgWaves = 8, kRgRows = 64, kRgPitch = kRgRows + 4;   // floats of a token's row in the exchange space: four rows apart, other banks
template <int TA> constexpr int kRgLds = 4 * TA * 16 * kRgPitch * int(sizeof(float));

// the gate row's logits of tokens [t0, t1) (zeros without a gate row), a wave a token; and the grid's share of what is to be cleared
template <int XT>
__device__ __forceinline__ void router_shared_column(const uint8_t * __restrict__ shared, const uint8_t * __restrict__ x, float * __restrict__ logits, int h, int e, int n,
                                                     int t0, int t1, const RouterSide & side, int waves) {
    const int lane = threadIdx.x & 63;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < side.zero_n; i += gridDim.x * blockDim.x) side.zero[i] = 0;
    for (int t = t0 + (threadIdx.x >> 6); t < t1; t += waves) {
        float acc = 0.f;
        if (shared)
            for (int c = lane * 8; c < h; c += 512) {
                float wv[8], xv[8];
                load8<XT>(shared, c, wv);
                load8<XT>(x, int64_t(t) * h + c, xv);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc = fmaf(wv[j], xv[j], acc);
            }
        acc = group_sum<64>(acc);
        if (lane == 0) logits[int64_t(t) * (e + 1) + e] = acc;
    }
}

// The same, in the same order, with the loads of several tokens and of four passes over its columns under way at once: one after the other
// they are a chain of trips to memory, longer than the blocks beside it where those are short or wait for it (us a launch, one after the other /
// so: 3500 tokens x 513 rows of 2048 32.3 / 21.4, 6000 x 61 of 4096 38.6 / 27.9, 8192 x 257 of 3072 38.4 / 35.6). Tokens and passes that are
// not there are branched around: as loads of zeros and of the last token again they cost 512 columns 7 %, two tokens a wave up to 17 %.
// The loop above stays where the gate row's blocks have time (launch_router_gemm), in the fp32 tiles straight from memory, whose main loop is
// slower with more code beside it (512 experts, 6000 tokens of 2048 166 / 174, 8192 of 1024 114 / 118), and in the kernel of large batches for
// blocks of the gate row's own that are all resident beside the others (8192 tokens x 129 rows of 7168 56.4 / 59.0, 5000 x 193 of 4096 35.3 / 36.3) and
// for shares of up to four passes a wave (8192 x 513 of 512 19.9 / 20.2, 3072 x 1001 of 768 24.0 / 25.2, 7168 x 701 of 640 31.4 / 32.7; longer ones
// gain: 8192 x 385 of 1024 29.7 / 27.8).
template <int XT>
__device__ __forceinline__ void router_shared_together(const uint8_t * __restrict__ shared, const uint8_t * __restrict__ x, float * __restrict__ logits, int h, int e, int n,
                                                     int t0, int t1, const RouterSide & side, int waves) {
    const int lane = threadIdx.x & 63;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < side.zero_n; i += gridDim.x * blockDim.x) side.zero[i] = 0;
    constexpr int NT = XT == TQMOE_F32 ? 2 : 4, NP = 4, RAW = XT == TQMOE_F32 ? 2 : 1, kSize = XT == TQMOE_F32 ? 4 : 2;   // tokens and passes together, loads of eight values
    for (int t = t0 + __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6); t < t1; t += NT * waves) {
        float acc[NT] = {};
        if (shared)
            for (int c0 = 0; c0 < h; c0 += NP * 512) {
                uint4 wr[NP][RAW], xr[NT][NP][RAW];
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const int c = c0 + p * 512 + lane * 8;          // (past the last column: zeros on both sides)
#pragma unroll
                    for (int q = 0; q < RAW; ++q) {
                        wr[p][q] = uint4();
#pragma unroll
                        for (int i = 0; i < NT; ++i) xr[i][p][q] = uint4();
                    }
                    if (c0 + p * 512 < h) {
                        if (c < h)
#pragma unroll
                            for (int q = 0; q < RAW; ++q) wr[p][q] = *reinterpret_cast<const uint4 *>(shared + int64_t(c) * kSize + q * 16);
#pragma unroll
                        for (int i = 0; i < NT; ++i)
                            if (t + i * waves < t1 && c < h)
#pragma unroll
                                for (int q = 0; q < RAW; ++q) xr[i][p][q] = *reinterpret_cast<const uint4 *>(x + (int64_t(t + i * waves) * h + c) * kSize + q * 16);
                    }
                }
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    if (c0 + p * 512 >= h) break;
                    float wv[8], xv[8];
                    load8<XT>(wr[p], 0, wv);
#pragma unroll
                    for (int i = 0; i < NT; ++i) {
                        if (t + i * waves >= t1) break;
                        load8<XT>(xr[i][p], 0, xv);
#pragma unroll
                        for (int j = 0; j < 8; ++j) acc[i] = fmaf(wv[j], xv[j], acc[i]);
                    }
                }
            }
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            if (t + i * waves >= t1) break;
            const float sum = group_sum<64>(acc[i]);
            if (lane == 0) logits[int64_t(t + i * waves) * (e + 1) + e] = sum;
        }
    }
}

// TOGETHER: the gate row's blocks have their loads together (launch_router_gemm says when)
template <bool F32, int TA, bool TOGETHER>
__global__ __launch_bounds__(64 * kRgWaves) void router_gemm_k(const uint8_t * __restrict__ w, const uint8_t * __restrict__ shared, const uint8_t * __restrict__ x,
                                                              float * __restrict__ logits, int h, int e, int n, RouterSide side) {
    extern __shared__ __attribute__((aligned(16))) float red[];   // [4][TA * 16][kRgPitch]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    constexpr int kBytes = F32 ? 4 : 2, TT = 16 * TA;
    const int t0 = int(blockIdx.x) * TT, r0 = int(blockIdx.y) * kRgRows;
    const int64_t pitch = int64_t(h) * kBytes;
    if (blockIdx.y == gridDim.y - 1) {
        if constexpr (TOGETHER) router_shared_together<F32 ? TQMOE_F32 : TQMOE_BF16>(shared, x, logits, h, e, n, t0, min(t0 + TT, n), side, kRgWaves);
        else router_shared_column<F32 ? TQMOE_F32 : TQMOE_BF16>(shared, x, logits, h, e, n, t0, min(t0 + TT, n), side, kRgWaves);
        return;
    }
    const uint8_t * ap[TA], * bp[4];   // rows past the end repeat a valid row (not stored)
#pragma unroll
    for (int i = 0; i < TA; ++i) ap[i] = x + int64_t(min(t0 + 16 * i + r, n - 1)) * pitch + 16 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) bp[j] = w + int64_t(min(r0 + 16 * j + r, e - 1)) * pitch + 16 * g;
    const int steps = int(pitch / 64), s0 = wave * steps / kRgWaves, s1 = (wave + 1) * steps / kRgWaves;   // 64 bytes of every row a step
    v4f acc[TA][4];
#pragma unroll
    for (int i = 0; i < TA; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    constexpr int C = TA == 4 ? 2 : 4;   // steps of loads together, and as many under way
    uint4 a[2][C][TA], b[2][C][4];
    auto fetch = [&](int st, int buf) {
        // (a row's steps one after the other: both halves of a 128-byte line before other rows' lines push it out of the first-level
        // cache. fp32, 64 experts, 4096 tokens: 30.4 -> 27.1 us; bf16 the same)
        int64_t at[C];
#pragma unroll
        for (int q = 0; q < C; ++q) at[q] = int64_t(min(st + q, s1 - 1)) * 64;
#pragma unroll
        for (int i = 0; i < TA; ++i)
#pragma unroll
            for (int q = 0; q < C; ++q) a[buf][q][i] = *reinterpret_cast<const uint4 *>(ap[i] + at[q]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < C; ++q) b[buf][q][j] = *reinterpret_cast<const uint4 *>(bp[j] + at[q]);
    };
    auto multiply = [&](int st, int buf) {
#pragma unroll
        for (int q = 0; q < C; ++q) {
            if (st + q >= s1) break;
#pragma unroll
            for (int i = 0; i < TA; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (F32) {   // lane group g's four columns with the other groups' four, one of each a time
                        const v4f av = __builtin_bit_cast(v4f, a[buf][q][i]), bv = __builtin_bit_cast(v4f, b[buf][q][j]);
#pragma unroll
                        for (int c = 0; c < 4; ++c) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[c], bv[c], acc[i][j], 0, 0, 0);
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[buf][q][i]), __builtin_bit_cast(v8bf, b[buf][q][j]), acc[i][j], 0, 0, 0);
                    }
                }
        }
    };
    if (s0 < s1) {
        fetch(s0, 0);
        for (int st = s0; st < s1; st += 2 * C) {
            if (st + C < s1) fetch(st + C, 1);
            multiply(st, 0);
            if (st + C >= s1) break;
            if (st + 2 * C < s1) fetch(st + 2 * C, 0);
            multiply(st + C, 1);
        }
    }
    // result register q of lane group g: token 4 g + q of the 16, router row r
    auto at = [&](int slot, int i, int q) { return (slot * TT + 16 * i + 4 * g + q) * kRgPitch + r; };
    if (wave >= 4) {
#pragma unroll
        for (int i = 0; i < TA; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) red[at(wave - 4, i, q) + 16 * j] = acc[i][j][q];
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int i = 0; i < TA; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) red[at(wave, i, q) + 16 * j] += acc[i][j][q];
    }
    __syncthreads();
    for (int i = tid; i < TT * kRgRows; i += 64 * kRgWaves) {
        const int t = i / kRgRows, c = i % kRgRows;
        const float * p = red + t * kRgPitch + c;
        const float v = (p[0] + p[TT * kRgPitch]) + (p[2 * TT * kRgPitch] + p[3 * TT * kRgPitch]);
        if (t0 + t < n && r0 + c < e) logits[int64_t(t0 + t) * (e + 1) + r0 + c] = v;
    }
}
// The same tile of 16 tokens x 64 router rows with every wave's operands through a place of its own in LDS: 128 bytes of a row, a whole
// line, in one transfer. With operands straight from memory an instruction touches sixteen rows, half a line each, and the lines of a wave's
// loads under way are many times the first-level cache: the loads ran at 15 bytes a cycle and compute unit, the first four waves' in front of
// the others' (333 tokens x 513 rows of 2048: waves 0 to 3 done after 11600 cycles, 4 to 7 after 21700). No wave waits for another before
// the partial tiles are added, in the same order: same bits. Two stages of 80 rows a wave are all of a compute unit's LDS.
// (us a launch, 2048 columns, operands from memory / so: bf16 333 tokens x 512 rows 11.8 / 7.5, with a 513th 11.7 / 7.4, 2100 x 64 11.5 / 7.5;
// fp32 333 x 512 24.3 / 16.2, 4096 x 64 27.4 / 20.5. All of a compute unit's LDS is one block's, so the gate row's blocks wait for a free one.)
constexpr int kRdRows = 16 + kRgRows, kRdStage = kRdRows * 128, kRdLds = kRgWaves * 2 * kRdStage;
static_assert(kRdLds <= 163840 && kRgLds<1> <= kRdLds, "the compute unit's LDS");
template <bool F32>
__global__ __launch_bounds__(64 * kRgWaves) void router_gemm_dma_k(const uint8_t * __restrict__ w, const uint8_t * __restrict__ shared, const uint8_t * __restrict__ x,
                                                                  float * __restrict__ logits, int h, int e, int n, int gate, RouterSide side) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];   // [wave][2][row][128]; then the partial tiles [4][16][kRgPitch]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    constexpr int kBytes = F32 ? 4 : 2, NQ = kRdRows / 8;
    const int t0 = int(blockIdx.x) * 16, r0 = int(blockIdx.y) * kRgRows;
    const int64_t pitch = int64_t(h) * kBytes;
    if (blockIdx.y == gridDim.y - 1) {
        router_shared_together<F32 ? TQMOE_F32 : TQMOE_BF16>(shared, x, logits, h, e, n, int(blockIdx.x) * gate, min(int(blockIdx.x + 1) * gate, n), side, kRgWaves);
        return;
    }
    // transfer q: rows 8 q .. + 7, the tokens' in front of the router's (past the end a valid row again, not stored); a row's 16-byte piece p
    // in slot p ^ (row / 2 & 7)
    const uint8_t * src[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int row = q * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
        src[q] = (row < 16 ? x + int64_t(min(t0 + row, n - 1)) * pitch : w + int64_t(min(r0 + row - 16, e - 1)) * pitch) + piece * 16;
    }
    const int steps = int(pitch / 64), s0 = wave * steps / kRgWaves, s1 = (wave + 1) * steps / kRgWaves;   // 64 bytes of every row a step, two a stage
    uint8_t * const own = lds + wave * 2 * kRdStage;
    const uint32_t own0 = lds_address(own);
    auto place = [&](int st) { return int(min(int64_t(st) * 64, pitch - 128)); };   // (an odd last step is a stage's second half)
    auto send = [&](int st, int slot) {
        const int at = place(st);
#pragma unroll
        for (int q = 0; q < NQ; ++q) dma16(src[q] + at, own0 + slot * kRdStage + q * 1024);
    };
    v4f acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    if (s0 < s1) {
        send(s0, 0);
        send(min(s0 + 2, s1 - 1), 1);
        int slot = 0;
        for (int st = s0; st < s1; st += 2, slot ^= 1) {
            dma_wait<NQ, false>();             // the other slot's may be under way
            const uint8_t * rows = own + slot * kRdStage + r * 128;
            const int skip = (st * 64 - place(st)) / 64;
            uint4 a[2], b[2][4];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int piece = ((4 * min(q + skip, 1) + g) ^ ((r >> 1) & 7)) * 16;   // (rows 16 further on have the same low bits)
                a[q] = *reinterpret_cast<const uint4 *>(rows + piece);
#pragma unroll
                for (int j = 0; j < 4; ++j) b[q][j] = *reinterpret_cast<const uint4 *>(rows + (16 + 16 * j) * 128 + piece);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            send(min(st + 4, s1 - 1), slot);   // (past the last stage: that one's last step again, not read)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (st + q >= s1) break;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (F32) {
                        const v4f av = __builtin_bit_cast(v4f, a[q]), bv = __builtin_bit_cast(v4f, b[q][j]);
#pragma unroll
                        for (int c = 0; c < 4; ++c) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[c], bv[c], acc[j], 0, 0, 0);
                    } else acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[q]), __builtin_bit_cast(v8bf, b[q][j]), acc[j], 0, 0, 0);
                }
            }
        }
    }
    dma_wait<0, true>();
    float * const red = reinterpret_cast<float *>(lds);
    auto at = [&](int slot, int q) { return (slot * 16 + 4 * g + q) * kRgPitch + r; };
    if (wave >= 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) red[at(wave - 4, q) + 16 * j] = acc[j][q];
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) red[at(wave, q) + 16 * j] += acc[j][q];
    }
    __syncthreads();
    for (int i = tid; i < 16 * kRgRows; i += 64 * kRgWaves) {
        const int t = i / kRgRows, c = i % kRgRows;
        const float * p = red + t * kRgPitch + c;
        const float v = (p[0] + p[16 * kRgPitch]) + (p[2 * 16 * kRgPitch] + p[3 * 16 * kRgPitch]);
        if (t0 + t < n && r0 + c < e) logits[int64_t(t0 + t) * (e + 1) + r0 + c] = v;
    }
}

// The same for large batches of bf16 rows: 64 tokens x 128 router rows a block, operands through LDS, so that a row of x is
// read by a quarter of the blocks. 128 bytes of every row a stage, from memory to LDS without registers, two stages under
// way, two blocks a compute unit. The eight parts of the columns follow each other and join in the order the kernel above adds them: same bits.
// (512 experts, 2048 columns, 4096 tokens: 24 us; 45 with every wave's operands from memory, 32 with stages of 512 bytes a
// row that pass registers.)
// Blocks from which it is the faster one (in us, this / operands from memory, 2048 columns: 64 blocks over 256 or 512 router
// rows 18.7 / 17.4, 128 blocks 19.2 / 27; 32 blocks 18.6 / 13.4; 1024 and 4096 columns cross at the same numbers). Up to 64
// router rows half the tile would be empty (60 rows, 4096 tokens: 18.6 / 13.5).
constexpr int kRlBlocks = 48;
constexpr int kRlFull = 224;    // blocks from which none are added for the gate row's column (256: 23 us against 31; 128: 32 against 19)
constexpr int kRlTok = 64, kRlRows = 128, kRlRing = 3, kRlStage = (kRlTok + kRlRows) * 128, kRlLds = kRlRing * kRlStage, kRlWaves = 8;
__global__ __launch_bounds__(64 * kRlWaves) void router_gemm_lds_k(const uint8_t * __restrict__ w, const uint8_t * __restrict__ shared, const uint8_t * __restrict__ x,
                                                         float * __restrict__ logits, int h, int e, int n, RouterSide side) {
    constexpr int NQ = (kRlTok + kRlRows) / 8 / kRlWaves;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int t0 = int(blockIdx.x) * kRlTok, r0 = int(blockIdx.y) * kRlRows;
    const int64_t pitch = int64_t(h) * 2;
    // The gate row's column: a last row of blocks where they find compute units free, else every block's share of its tokens.
    const int cols = (e + kRlRows - 1) / kRlRows;
    if (int(blockIdx.y) == cols) {
        if (gridDim.x * gridDim.y > 256) router_shared_together<TQMOE_BF16>(shared, x, logits, h, e, n, t0, min(t0 + kRlTok, n), side, kRlWaves);
        else router_shared_column<TQMOE_BF16>(shared, x, logits, h, e, n, t0, min(t0 + kRlTok, n), side, kRlWaves);
        return;
    }
    // transfer q of a wave is eight rows of a stage: the tokens' rows, then the router's; a row's 16-byte piece p in slot
    // p ^ (row / 2 & 7)
    const uint8_t * src[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int row = (NQ * wave + q) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
        src[q] = (row < kRlTok ? x + int64_t(min(t0 + row, n - 1)) * pitch : w + int64_t(min(r0 + row - kRlTok, e - 1)) * pitch) + piece * 16;
    }
    const uint32_t lds0 = lds_address(lds);
    const int steps = int(pitch / 64);
    auto part_of = [&](int k) { return (k & 1) * 4 + (k >> 1); };          // parts 0, 4, 1, 5, 2, 6, 3, 7
    auto first = [&](int k) { return part_of(k) * steps / kRgWaves; };
    auto last = [&](int k) { return (part_of(k) + 1) * steps / kRgWaves; };
    int sk = 0, ss = first(0), slot_in = 0;                                // the next stage to send
    while (sk < 8 && ss >= last(sk)) { ++sk; ss = sk < 8 ? first(sk) : 0; }
    auto send = [&]() {
        if (sk < 8) {
            const int64_t at = min(int64_t(ss) * 64, pitch - 128);        // (a part's odd last step: half a stage is not used)
#pragma unroll
            for (int q = 0; q < NQ; ++q) dma16(src[q] + at, lds0 + slot_in * kRlStage + (NQ * wave + q) * 1024);
            ss += 2;
            while (sk < 8 && ss >= last(sk)) { ++sk; ss = sk < 8 ? first(sk) : 0; }
        }
        slot_in = slot_in + 1 == kRlRing ? 0 : slot_in + 1;
    };
    int total = 0;
    for (int k = 0; k < 8; ++k) total += (last(k) - first(k) + 1) / 2;
#pragma unroll
    for (int i = 0; i < kRlRing - 1; ++i) send();
    if (int(gridDim.y) == cols) {   // (under the first transfers)
        const int share = (kRlTok + cols - 1) / cols, first_t = t0 + int(blockIdx.y) * share;
        const int last_t = min(min(first_t + share, t0 + kRlTok), n);
        if (h > 512 && share * ((h + 511) / 512) > 32) router_shared_together<TQMOE_BF16>(shared, x, logits, h, e, n, first_t, last_t, side, kRlWaves);
        else router_shared_column<TQMOE_BF16>(shared, x, logits, h, e, n, first_t, last_t, side, kRlWaves);
    }
    const int tq = wave & 1, rq = wave >> 1;
    const uint8_t * a_row = lds + (tq * 32 + r) * 128, * b_row = lds + (kRlTok + rq * 32 + r) * 128;
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f acc[2][2], pair[2][2], half[2][2], sum[2][2];
    int slot = 0, done = 0;
    for (int k = 0; k < 8; ++k) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = zero;
        for (int st = first(k); st < last(k); st += 2) {
            if (done + kRlRing - 1 <= total) dma_wait<NQ * (kRlRing - 2), true>(); else dma_wait<0, true>();
            send();
            const int skip = int64_t(st) * 64 > pitch - 128 ? 1 : 0;      // the step is the stage's second half
            const uint8_t * as = a_row + slot * kRlStage, * bs = b_row + slot * kRlStage;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (q == 1 && st + 1 >= last(k)) break;
                const int piece = (4 * (q + skip) + g) ^ ((r >> 1) & 7);   // (rows 16 further on have the same low bits)
                v8bf a[2], b[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[i] = *reinterpret_cast<const v8bf *>(as + i * 2048 + piece * 16);
                    b[i] = *reinterpret_cast<const v8bf *>(bs + i * 2048 + piece * 16);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
            }
            slot = slot + 1 == kRlRing ? 0 : slot + 1;
            ++done;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if ((k & 1) == 0) pair[i][j] = acc[i][j];
                else {
                    pair[i][j] += acc[i][j];
                    if (k == 1 || k == 5) half[i][j] = pair[i][j];
                    else if (k == 3) sum[i][j] = half[i][j] + pair[i][j];
                    else sum[i][j] = sum[i][j] + (half[i][j] + pair[i][j]);
                }
            }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int t = t0 + tq * 32 + 16 * i + 4 * g + q, c = r0 + rq * 32 + 16 * j + r;
                if (t < n && c < e) logits[int64_t(t) * (e + 1) + c] = sum[i][j][q];
            }
}
template <bool F32> void launch_router_gemm(const void * w, const void * sg, const void * x, float * logits, int h, int e, int n, const RouterSide & side, hipStream_t s) {
    const int64_t rows = (e + kRgRows - 1) / kRgRows;
    auto blocks = [&](int ta) { return ((n + 16 * ta - 1) / (16 * ta)) * rows; };
    auto go = [&](auto tile) {
        constexpr int TA = decltype(tile)::value;
        const int tiles = (n + 16 * TA - 1) / (16 * TA);
        auto kernel = &router_gemm_k<F32, TA, false>;
        // The gate row's blocks have their loads together where they open another round of the compute units. Beside the last one they have its
        // time, and together take from its blocks' bandwidth (bf16, us, one after the other / together: 256 blocks of 64 tokens and 128 of the
        // gate row 19.9 / 17.0, 440 and 55 42.4 / 43.3, 128 and 128 32.8 / 34.4).
        if constexpr (!F32)
            if ((blocks(TA) - 1) % 256 + 1 + tiles > 256) kernel = &router_gemm_k<F32, TA, true>;
        allow_dynamic_lds(reinterpret_cast<const void *>(kernel), kRgLds<TA>);
        kernel<<<dim3(unsigned(tiles), unsigned(rows + 1)), 64 * kRgWaves, kRgLds<TA>, s>>>(
            static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(sg), static_cast<const uint8_t *>(x), logits, h, e, n, side);
    };
    const bool aligned = aligned16(w) && aligned16(x), long_rows = int64_t(h) * (F32 ? 4 : 2) >= 4096;
    auto rounds = [&](int ta) { return (blocks(ta) + 255) / 256; };
    // (operands through LDS / straight from memory. Where straight would be tiles of 16 tokens: 1024 columns, 200 tokens x 512 rows,
    // 5.4 / 7.2 us, 512 columns 4.7 / 7.2, 128 4.0 / 4.9; fp32 9.5 / 13.3, 6.8 / 7.8, 4.9 / 7.2. Of more blocks long rows only; bf16, us
    // beside tiles of 32 tokens, 256 blocks of 16: 2048 columns 11.6 / 14.1, 4096 15.0 / 24.1, but 1024 9.2 / 8.6; 64 experts, 375 blocks:
    // 1024 columns 12.8 / 9.0, 4096 26.1 / 27.0; beside the kernel of large batches, 384, 512 and 768 blocks: 2048 columns 14.1 / 19.1, 16.8 /
    // 19.1, 24.2 / 19.6, 1024 columns 11.0 / 12.2, 14.2 / 12.3. fp32, beside 32 tokens, 512 and 768 blocks: 2048 columns 32.0 / 39.0, 46.1 / 65.0,
    // 1024 18.8 / 22.0, 27.0 / 36.4, but 512 13.7 / 13.0; beside 64 tokens, a round of 256 blocks, one and a half, two: 2048 columns 60 / 60,
    // 88 / 110, 120 / 115, 1024 35 / 32, 52 / 53, 70 / 59; by rounds of 16 and of 64 tokens, 1024 columns, 7 and 2 59.7 / 59.9, 10 and 3 84.5 / 87.1,
    // 14 and 4 119 / 109, 2048 columns 14 and 4 197 / 211; 10 and 3, fewer experts: 1024 columns, 8192 tokens x 320 86.9 / 81.3, 10000 x 256 88.0 / 83.2, but
    // 1792 columns 134 / 153, 136 / 156)
    if (aligned && (F32 ? blocks(2) < 256 || (long_rows && (blocks(4) < 256 || (h >= 2048 ? 11 * rounds(1) < 40 * rounds(4) : h > 1024 ? 5 * rounds(1) < 17 * rounds(4) : 3 * rounds(1) < 10 * rounds(4))))
                        : blocks(2) < 128 || (long_rows && blocks(1) <= (e > kRgRows ? 512 : 256)))) {
        // a block of the gate row's takes 32 tokens instead of 16 where all of short rows' blocks nearly fit the chip at once (64 experts, 1024
        // columns: 2100 tokens 5.9 us against 6.4, 3072 7.0 against 8.4; 2048 columns 8.1 against 7.4, and fp32 no better either)
        const unsigned tiles = unsigned((n + 15) / 16);
        const int gate = !F32 && !long_rows && blocks(1) <= 256 && blocks(1) + tiles > 256 ? 32 : 16;
        allow_dynamic_lds(reinterpret_cast<const void *>(&router_gemm_dma_k<F32>), kRdLds);
        router_gemm_dma_k<F32><<<dim3(tiles, unsigned(rows + 1)), 64 * kRgWaves, kRdLds, s>>>(
            static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(sg), static_cast<const uint8_t *>(x), logits, h, e, n, gate, side);
        return;
    }
    if constexpr (!F32) {
        const int64_t tiles = (n + kRlTok - 1) / kRlTok, cols = (e + kRlRows - 1) / kRlRows;
        if (tiles * cols >= kRlBlocks && e > kRgRows && h >= 512 && aligned) {
            allow_dynamic_lds(reinterpret_cast<const void *>(&router_gemm_lds_k), kRlLds);
            router_gemm_lds_k<<<dim3(unsigned(tiles), unsigned(cols + (tiles * cols < kRlFull ? 1 : 0))), 64 * kRlWaves, kRlLds, s>>>(
                static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(sg), static_cast<const uint8_t *>(x), logits, h, e, n, side);
            return;
        }
    }
    // (2048 columns, us with 16 / 32 / 64 tokens a block: bf16, 128 blocks of 32 tokens 14.9 / 13.5 / 17.6, 128 of 64 28 / 21 / 19; fp32, 128
    // blocks of 32 tokens 27 / 43 / 71, 256 of 64 106 / 85 / 79)
    if (blocks(4) >= (F32 ? 256 : 128)) go(std::integral_constant<int, 4>{});
    else if (blocks(2) >= (F32 ? 256 : 128)) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 1>{});
}

// ------------------------------------------------------------------------------------------------------ top-k
// One wave per token. Selection rule of the reference: larger probability first, equal probabilities to the lower
// index. Up to 1024 experts the probabilities stay in registers (lane l owns entries l, l + 64, ...) and every
// reduction is a DPP butterfly ending in a scalar broadcast; larger layers keep them in LDS.
struct TopkOut {
    int * ids; float * weights; float * shared_weights;
    int * ext_ids; int extra;          // optional [n][k + 1] copy of the ids with `extra` in the last slot
    int shared_ungated;                // the shared expert has no gate row: its weight is 1, not sigmoid(0)
    TopkSide side;
};
__device__ __forceinline__ float shared_weight_of(const TopkOut & o, float logit) { return o.shared_ungated ? 1.f : 1.f / (1.f + expf(-logit)); }

__device__ __forceinline__ void topk_finish(const TopkOut & o, const float * x_logits, int token, int lane, int e, int k, float scale, float selected) {
    if (lane == 0) {
        const float total = fmaxf(selected, 6.103515625e-5f);
        for (int s = 0; s < k; ++s) {   // the host divides by the clamped sum, then multiplies by the scale
            float v = o.weights[int64_t(token) * k + s] / total;
            if (scale != 0.f && scale != 1.f) v *= scale;
            o.weights[int64_t(token) * k + s] = v;
        }
        if (o.shared_weights) o.shared_weights[token] = shared_weight_of(o, x_logits[e]);
        if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + k] = o.extra;
    }
}

// the token's input row in the form the products read
template <int XT> __device__ __forceinline__ void topk_row(const TopkOut & o, int token, int lane) {
    const TopkSide & d = o.side;
    switch (d.rows) {
        case kRowsImage: quantise_row_wave<XT>(d.x, token, d.cols, static_cast<uint8_t *>(d.q) + int64_t(token) * (d.cols / 32) * kImageSubBytes, lane); break;
        case kRowsHalves: prepare_row_wave<XT>(d.x, token, d.cols, static_cast<uint16_t *>(d.q), d.scale, lane); break;
        case kRowsFp8: quant_row_wave<XT, true, false>(d.x, token, d.cols, static_cast<int8_t *>(d.q), d.scale, nullptr, lane); break;
        case kRowsInt8: quant_row_wave<XT, false, false>(d.x, token, d.cols, static_cast<int8_t *>(d.q), d.scale, nullptr, lane); break;
        case kRowsInt8Blocks: quant_row_wave<XT, false, true>(d.x, token, d.cols, static_cast<int8_t *>(d.q), d.scale, nullptr, lane); break;
    }
}
// selection s of the token is expert id (s = k: the shared one): one more assignment of it in the dispatch chunk. An id
// outside the banks is not counted, as the dispatch that reads the counts does not place it.
__device__ __forceinline__ void topk_count(const TopkOut & o, int token, int k, int s, int id) {
    if (!o.side.chunk_counts || id < 0 || id >= o.side.banks) return;
    const int64_t a = int64_t(token) * (o.ext_ids ? k + 1 : k) + s;
    atomicAdd(o.side.chunk_counts + a / kDispatchChunk * o.side.banks + id, 1);
}

// With rows to write the block has a second wave that does nothing else: the row's quantisation runs beside the selection
// instead of after it.
template <int R, int XT>
__device__ __forceinline__ void topk_reg_body(const float * __restrict__ logits, const TopkOut & o, int e, int k, float scale) {
    const int token = blockIdx.x, lane = threadIdx.x & 63;
    const float * x = logits + int64_t(token) * (e + 1);
    if (threadIdx.x >= 64) {
        topk_row<XT>(o, token, lane);
        return;
    }
    const float shared_logit = o.shared_weights ? x[e] : 0.f;
    if (k <= 64) {
        int my_id;
        float my_w;
        __shared__ __attribute__((aligned(16))) int cand[256];
        topk_select<R>(topk_logits<R>(x, e, lane), e, k, lane, true, cand, my_id, my_w);
        const float v = topk_weight(my_w, k, scale);
        if (lane < k) {
            o.ids[int64_t(token) * k + lane] = my_id;
            o.weights[int64_t(token) * k + lane] = v;
            if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + lane] = my_id;
            topk_count(o, token, k, lane, my_id);
        }
        if (lane == 0) {
            if (o.shared_weights) o.shared_weights[token] = shared_weight_of(o, shared_logit);
            if (o.ext_ids) { o.ext_ids[int64_t(token) * (k + 1) + k] = o.extra; topk_count(o, token, k, k, o.extra); }
        }
        return;
    }
    // more selections than lanes
    int key[R];
    float m = -INFINITY, sum = 0.f;
    {
        float l[R];
#pragma unroll
        for (int r = 0; r < R; ++r) { const int j = lane + 64 * r; l[r] = j < e ? x[j] : -INFINITY; m = fmaxf(m, l[r]); }
        m = wave_max_all(m);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int j = lane + 64 * r;
            const float ex = j < e ? expf(l[r] - m) : 0.f;
            sum += ex;
            key[r] = j < e ? (ex > 0.f ? order_key(l[r]) : kKeyZero) : kKeyGone;   // entries past the end never win
        }
        sum = wave_sum_all(sum);
    }
    float selected = 0.f, my_w = 0.f;   // lane s keeps selection s
    int my_id = 0;
    for (int s = 0; s < k; ++s) {
        int bk = key[0], bi = lane;
#pragma unroll
        for (int r = 1; r < R; ++r) if (key[r] > bk) { bk = key[r]; bi = lane + 64 * r; }   // strict: the lowest index of equal keys
        const int topkey = wave_max_all_i(bk);
        const int best = wave_min_all(bk == topkey ? bi : 0x7FFFFFFF);
        const float top = topkey == kKeyZero ? 0.f : expf(key_value(topkey) - m) / sum;   // the probability, as every entry's would be computed
        if (lane == (s & 63)) { my_id = best; my_w = top; }
        if ((s & 63) == 63) {   // a full set goes out before the lanes are reused
            o.ids[int64_t(token) * k + s - 63 + lane] = my_id;
            o.weights[int64_t(token) * k + s - 63 + lane] = my_w;   // divided below
            if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + s - 63 + lane] = my_id;
        }
        selected += top;                       // slot order, as the host sums the selected weights
#pragma unroll
        for (int r = 0; r < R; ++r) if (lane + 64 * r == best) key[r] = kKeyGone;
    }
    const int done = k & ~63;             // the last partial set
    if (lane < k - done) {
        o.ids[int64_t(token) * k + done + lane] = my_id;
        o.weights[int64_t(token) * k + done + lane] = my_w;
        if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + done + lane] = my_id;
    }
    __threadfence_block();
    topk_finish(o, x, token, lane, e, k, scale, selected);
}

template <int R, int XT>
__global__ __launch_bounds__(128) void topk_reg_k(const float * __restrict__ logits, TopkOut o, int e, int k, float scale) {
    topk_reg_body<R, XT>(logits, o, e, k, scale);
}
// two routings of the same shape in one launch (blockIdx.y picks): this layer's and a prediction of the next layer's
template <int R>
__global__ __launch_bounds__(64) void topk2_reg_k(const float * __restrict__ logits, TopkOut o, const float * __restrict__ logits2, TopkOut o2, int e, int k,
                                                  float scale) {
    if (blockIdx.y == 0) topk_reg_body<R, TQMOE_F32>(logits, o, e, k, scale);
    else topk_reg_body<R, TQMOE_F32>(logits2, o2, e, k, scale);
}

template <int XT>
__global__ __launch_bounds__(64) void topk_lds_k(const float * __restrict__ logits, TopkOut o, int e, int k, float scale) {
    extern __shared__ int keys[];
    const int token = blockIdx.x, lane = threadIdx.x;
    const float * x = logits + int64_t(token) * (e + 1);
    float m = -INFINITY;
    for (int j = lane; j < e; j += 64) m = fmaxf(m, x[j]);
    m = wave_max_all(m);
    float sum = 0.f;
    for (int j = lane; j < e; j += 64) { const float ex = expf(x[j] - m); keys[j] = ex > 0.f ? order_key(x[j]) : kKeyZero; sum += ex; }
    sum = wave_sum_all(sum);
    float selected = 0.f;
    for (int s = 0; s < k; ++s) {
        int bk = kKeyGone, bi = 0x7FFFFFFF;
        for (int j = lane; j < e; j += 64) if (keys[j] > bk) { bk = keys[j]; bi = j; }
        const int topkey = wave_max_all_i(bk);
        const int best = wave_min_all(bk == topkey ? bi : 0x7FFFFFFF);
        const float top = topkey == kKeyZero ? 0.f : expf(key_value(topkey) - m) / sum;
        if (lane == 0) {
            o.ids[int64_t(token) * k + s] = best;
            o.weights[int64_t(token) * k + s] = top;
            if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + s] = best;
        }
        selected += top;
        if ((best & 63) == lane) keys[best] = kKeyGone;
    }
    topk_finish(o, x, token, lane, e, k, scale, selected);
    if (o.side.rows) topk_row<XT>(o, token, lane);
}

template <int XT> void launch_topk(const float * logits, const TopkOut & o, int e, int k, int n, float scale, hipStream_t s) {
    if (e <= 64) topk_reg_k<1, XT><<<unsigned(n), o.side.rows ? 128 : 64, 0, s>>>(logits, o, e, k, scale);
    else if (e <= 128) topk_reg_k<2, XT><<<unsigned(n), o.side.rows ? 128 : 64, 0, s>>>(logits, o, e, k, scale);
    else if (e <= 256) topk_reg_k<4, XT><<<unsigned(n), o.side.rows ? 128 : 64, 0, s>>>(logits, o, e, k, scale);
    else if (e <= 512) topk_reg_k<8, XT><<<unsigned(n), o.side.rows ? 128 : 64, 0, s>>>(logits, o, e, k, scale);
    else if (e <= 1024) topk_reg_k<16, XT><<<unsigned(n), o.side.rows ? 128 : 64, 0, s>>>(logits, o, e, k, scale);
    else topk_lds_k<XT><<<unsigned(n), 64, size_t(e) * sizeof(float), s>>>(logits, o, e, k, scale);
}

// The reference's other gating functions (src/experts/moe.cpp:22-113): sigmoid, softmax over the selected logits only,
// sqrt(softplus); a selection bias added for the choice but not for the weights; weights left unnormalised on request.
// One wave per token as above; the values of lane's experts (lane, lane + 64, ...) sit in registers for up to 1024
// experts and in LDS beyond. A taken mask replaces the "below every value" marker of the softmax kernel, since biased
// values and raw logits have no lower bound.
struct Gate { const float * bias; int gating, norm; };

__device__ __forceinline__ float gate_value(int gating, float x) {
    if (gating == TQMOE_GATE_SIGMOID) return 1.0f / (1.0f + expf(-x));
    if (gating == TQMOE_GATE_SQRT_SOFTPLUS) return sqrtf(x > 0.f ? x + log1pf(expf(-x)) : log1pf(expf(x)));
    return x;   // softmax over the selection: the logits themselves
}

// lane 0 finishes a token with more selections than lanes from the raw weights in memory, in slot order as the host does
__device__ void gated_finish_serial(float * w, int k, const Gate & g, float scale) {
    if (g.gating == TQMOE_GATE_SOFTMAX_WEIGHT) {
        float mx = -INFINITY, sum = 0.f;
        for (int s = 0; s < k; ++s) mx = fmaxf(mx, w[s]);
        for (int s = 0; s < k; ++s) { w[s] = expf(w[s] - mx); sum += w[s]; }
        for (int s = 0; s < k; ++s) w[s] = w[s] / sum;
    }
    if (g.norm) {
        float sum = 0.f;
        for (int s = 0; s < k; ++s) sum += w[s];
        sum = fmaxf(sum, 6.103515625e-5f);
        for (int s = 0; s < k; ++s) w[s] = w[s] / sum;
    }
    if (scale != 0.f && scale != 1.f) for (int s = 0; s < k; ++s) w[s] *= scale;
}

// sum over lanes 0 .. k - 1 in lane order (the host's slot order), k <= 64
__device__ __forceinline__ float slot_order_sum(float v, int k) {
    float sum = 0.f;
    for (int s = 0; s < k; ++s) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), s));
    return sum;
}

template <int R, int XT>   // R = 0: values in LDS, ceil(e / 64) per lane
__global__ __launch_bounds__(64) void topk_gated_k(const float * __restrict__ logits, TopkOut o, Gate g, int e, int k, float scale) {
    extern __shared__ float gated_lds[];
    constexpr bool kLds = R == 0;
    constexpr int kRegs = kLds ? 1 : R;
    const int token = blockIdx.x, lane = threadIdx.x;
    const float * x = logits + int64_t(token) * (e + 1);
    const int per_lane = kLds ? (e + 63) / 64 : R;
    float p_reg[kRegs], v_reg[kRegs];
    float * p_lds = gated_lds + lane, * v_lds = gated_lds + 64 * per_lane + lane;   // entry r of a lane at [64 r]: no bank conflicts
    auto P = [&](int r) -> float & { if constexpr (kLds) return p_lds[64 * r]; else return p_reg[r]; };
    auto V = [&](int r) -> float & { if constexpr (kLds) return v_lds[64 * r]; else return v_reg[r]; };

    const float shared_logit = o.shared_weights ? x[e] : 0.f;
    float m = -INFINITY;
#pragma unroll
    for (int r = 0; r < per_lane; ++r) { const int j = lane + 64 * r; P(r) = j < e ? x[j] : -INFINITY; m = fmaxf(m, P(r)); }
    if (g.gating == TQMOE_GATE_SOFTMAX) {
        m = wave_max_all(m);
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < per_lane; ++r) { const int j = lane + 64 * r; P(r) = j < e ? expf(P(r) - m) : 0.f; sum += P(r); }
        sum = wave_sum_all(sum);
#pragma unroll
        for (int r = 0; r < per_lane; ++r) P(r) = P(r) / sum;
    } else {
#pragma unroll
        for (int r = 0; r < per_lane; ++r) P(r) = gate_value(g.gating, P(r));
    }
#pragma unroll
    for (int r = 0; r < per_lane; ++r) {   // a NaN compares with nothing: it is chosen as the lowest value, so that every round finds an expert not yet taken
        const int j = lane + 64 * r;
        const float v = g.bias && j < e ? P(r) + g.bias[j] : P(r);
        V(r) = v == v ? v : -INFINITY;
    }
    uint64_t taken = 0;   // bit r: entry r of this lane is chosen already or lies past the end
#pragma unroll
    for (int r = 0; r < per_lane; ++r) if (lane + 64 * r >= e) taken |= uint64_t(1) << r;

    float selected = 0.f, my_w = 0.f;   // lane s keeps selection s
    int my_id = 0;
    for (int s = 0; s < k; ++s) {
        float bv = -INFINITY;
        int bi = 0x7FFFFFFF;
#pragma unroll
        for (int r = 0; r < per_lane; ++r)   // strict: the lowest index of equal values
            if (!(taken >> r & 1) && (bi == 0x7FFFFFFF || V(r) > bv)) { bv = V(r); bi = lane + 64 * r; }
        const float top = wave_max_all(bv);
        const int best = wave_min_all(bv == top && bi != 0x7FFFFFFF ? bi : 0x7FFFFFFF);
        float wv = 0.f;
#pragma unroll
        for (int r = 0; r < per_lane; ++r) if (lane + 64 * r == best) { wv = P(r); taken |= uint64_t(1) << r; }
        const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wv), best & 63));   // the unbiased value
        if (lane == (s & 63)) { my_id = best; my_w = w; }
        if (k > 64 && (s & 63) == 63) {   // more selections than lanes: a full set goes out before the lanes are reused
            o.ids[int64_t(token) * k + s - 63 + lane] = my_id;
            o.weights[int64_t(token) * k + s - 63 + lane] = my_w;
            if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + s - 63 + lane] = my_id;
        }
        selected += w;   // slot order, as the host sums the selected weights
    }
    if (k <= 64) {
        if (g.gating == TQMOE_GATE_SOFTMAX_WEIGHT) {
            const float mx = wave_max_all(lane < k ? my_w : -INFINITY);
            my_w = lane < k ? expf(my_w - mx) : 0.f;
            my_w = my_w / slot_order_sum(my_w, k);
            selected = slot_order_sum(my_w, k);
        }
        if (g.norm) my_w = my_w / fmaxf(selected, 6.103515625e-5f);
        if (scale != 0.f && scale != 1.f) my_w *= scale;
        if (lane < k) {
            o.ids[int64_t(token) * k + lane] = my_id;
            o.weights[int64_t(token) * k + lane] = my_w;
            if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + lane] = my_id;
            topk_count(o, token, k, lane, my_id);
        }
    } else {
        const int done = k & ~63;             // the last partial set
        if (lane < k - done) {
            o.ids[int64_t(token) * k + done + lane] = my_id;
            o.weights[int64_t(token) * k + done + lane] = my_w;
            if (o.ext_ids) o.ext_ids[int64_t(token) * (k + 1) + done + lane] = my_id;
        }
        __threadfence_block();
        if (lane == 0) gated_finish_serial(o.weights + int64_t(token) * k, k, g, scale);
    }
    if (lane == 0) {
        if (o.shared_weights) o.shared_weights[token] = shared_weight_of(o, shared_logit);
        if (o.ext_ids) { o.ext_ids[int64_t(token) * (k + 1) + k] = o.extra; topk_count(o, token, k, k, o.extra); }
    }
    if (o.side.rows) topk_row<XT>(o, token, lane);
}

template <int XT> void launch_topk_gated(const float * logits, const TopkOut & o, const Gate & g, int e, int k, int n, float scale, hipStream_t s) {
    if (e <= 64) topk_gated_k<1, XT><<<unsigned(n), 64, 0, s>>>(logits, o, g, e, k, scale);
    else if (e <= 128) topk_gated_k<2, XT><<<unsigned(n), 64, 0, s>>>(logits, o, g, e, k, scale);
    else if (e <= 256) topk_gated_k<4, XT><<<unsigned(n), 64, 0, s>>>(logits, o, g, e, k, scale);
    else if (e <= 512) topk_gated_k<8, XT><<<unsigned(n), 64, 0, s>>>(logits, o, g, e, k, scale);
    else if (e <= 1024) topk_gated_k<16, XT><<<unsigned(n), 64, 0, s>>>(logits, o, g, e, k, scale);
    else topk_gated_k<0, XT><<<unsigned(n), 64, size_t((e + 63) / 64) * 128 * sizeof(float), s>>>(logits, o, g, e, k, scale);
}

// --------------------------------------------------------------------------------------------------- dispatch
// Stable counting sort of the assignments by expert. Chunks of kChunk consecutive assignments; pass 1 counts each
// chunk's experts in LDS, pass 2 turns the per-chunk counts into exclusive prefixes (and counts / offsets), pass 3
// places every assignment at offsets[e] + prefix[chunk][e] + its rank among the chunk's earlier assignments of the
// same expert. Ranks come from ballots (lower lanes of the same expert) and a per-expert running count in LDS that
// waves add to in wave order, so no ordering is left to atomics. A single chunk runs all three passes in one block.
constexpr int kChunk = kDispatchChunk;

__device__ __forceinline__ void zero_lds(int * a, int n) {
    for (int j = threadIdx.x; j < n; j += blockDim.x) a[j] = 0;
}

// exclusive scan over e of run[0..E) into out[0..E], out[E] = total; one block, E <= 4096, scratch >= blockDim ints
__device__ void block_exclusive_scan(const int * run, int * out, int E, int * scratch) {
    const int tid = threadIdx.x, nt = blockDim.x;
    const int per = (E + nt - 1) / nt, lo = min(tid * per, E), hi = min(lo + per, E);
    int s = 0;
    for (int j = lo; j < hi; ++j) s += run[j];
    scratch[tid] = s;
    __syncthreads();
    for (int d = 1; d < nt; d <<= 1) {  // Hillis-Steele inclusive scan of the per-thread sums
        const int v = tid >= d ? scratch[tid - d] : 0;
        __syncthreads();
        scratch[tid] += v;
        __syncthreads();
    }
    int base = tid ? scratch[tid - 1] : 0;
    for (int j = lo; j < hi; ++j) { out[j] = base; base += run[j]; }
    if (tid == nt - 1) out[E] = scratch[nt - 1];
    __syncthreads();
}

__global__ __launch_bounds__(256) void dispatch_count_k(const int * __restrict__ ids, int * __restrict__ chunk_counts, int A, int E) {
    extern __shared__ int hist[];
    zero_lds(hist, E);
    __syncthreads();
    const int base = blockIdx.x * kChunk;
    for (int i = threadIdx.x; i < kChunk; i += 256) {
        const int a = base + i;
        if (a < A) { const int e = ids[a]; if (e >= 0 && e < E) atomicAdd(&hist[e], 1); }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < E; j += 256) chunk_counts[int64_t(blockIdx.x) * E + j] = hist[j];
}

__global__ __launch_bounds__(1024) void dispatch_scan_k(int * __restrict__ chunk_counts, int * __restrict__ counts,
                                                       int * __restrict__ offsets, int chunks, int E) {
    extern __shared__ int sm[];  // E totals, then 1024 scratch
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        int run = 0;
        for (int b = 0; b < chunks; ++b) {
            const int v = chunk_counts[int64_t(b) * E + e];
            chunk_counts[int64_t(b) * E + e] = run;
            run += v;
        }
        sm[e] = run;
        counts[e] = run;
    }
    __syncthreads();
    block_exclusive_scan(sm, offsets, E, sm + E);
}

// places one chunk; run[] = per-expert running count inside the chunk (LDS, zeroed by the caller)
__device__ void place_chunk(const int * __restrict__ ids, const int * __restrict__ offsets, const int * __restrict__ prefix,
                            int * __restrict__ perm, int * __restrict__ groups, int capacity, int base, int A, int E, int * run) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    for (int i0 = 0; i0 < kChunk && base + i0 < A; i0 += blockDim.x) {
        const int a = base + i0 + threadIdx.x;
        int e = a < A ? ids[a] : -1;
        if (e >= E) e = -1;
        // rank of this lane among the wave's earlier lanes of the same expert, and the size of its group
        int rank = 0, size = 0;
        bool last = false;
        unsigned long long todo = __ballot(e >= 0);
        while (todo) {
            const int leader = __ffsll(todo) - 1;
            const int v = __shfl(e, leader, 64);
            const unsigned long long same = __ballot(e == v);
            if (e == v) {
                rank = __popcll(same & ((1ull << lane) - 1ull));
                size = __popcll(same);
                last = (63 - __clzll(same)) == lane;
            }
            todo &= ~same;
        }
        for (int w = 0; w < waves; ++w) {  // waves take their turn in index order
            if (wave == w && e >= 0) {
                const int slot = (prefix ? prefix[e] : 0) + run[e] + rank;
                if (perm) perm[offsets[e] + slot] = a;
                if (groups && slot < capacity) groups[int64_t(e) * capacity + slot] = a;
            }
            __syncthreads();
            if (wave == w && e >= 0 && last) run[e] += size;
            __syncthreads();
        }
    }
}

__global__ __launch_bounds__(256) void dispatch_place_k(const int * __restrict__ ids, const int * __restrict__ offsets,
                                                        const int * __restrict__ chunk_prefix, int * __restrict__ perm,
                                                        int * __restrict__ groups, int capacity, int A, int E) {
    extern __shared__ int run[];
    zero_lds(run, E);
    __syncthreads();
    place_chunk(ids, offsets, chunk_prefix + int64_t(blockIdx.x) * E, perm, groups, capacity, blockIdx.x * kChunk, A, E, run);
}

// Pass 2 and 3 in one launch for up to kWideExperts experts: a block of sixteen waves takes a chunk, one wave per 64
// consecutive assignments, and thread j keeps expert j's sums. Every block adds up the per-chunk counts itself (the chunks
// before it: where its assignments start inside each expert; all chunks: the experts' offsets); a wave finds each lane's equals
// with a ballot per bit of the expert's number (a loop over the distinct experts of a wave's 64 assignments is 64 rounds at
// worst), leaves its group sizes in a histogram of its own, and a prefix over the waves in index order gives every
// assignment its place. Nothing is left to the order of atomics. One block more writes the counts and plans the products' items where it
// finds a compute unit of its own (behind its placement the first chunk's was the launch's longest; without items, and from 256 chunks on, that
// one does it). Prefix sums go through DPP and not through LDS a step at a time.
// Chunk counts are loaded sixteen at a time, without a look at their end but in the last sixteen (twenty-four, past the end the last one
// again, are half as many loads more than 16 or 32 chunks need and their addresses more scalar arithmetic than many chunks' loads take). Two
// blocks a compute unit, or more than 256 chunks are two rounds of them: 93 scalar and 64 vector registers were one block.
// us a launch, with the plan behind a placement, shuffles and a branch a load / a block for the plan, DPP and twenty-four / so: 333 tokens of 10
// of 512 experts 7.4 / 5.0 / 5.3, 1501 9.0 / 6.2 / 5.4, 4096 10.9 / 9.3 / 8.2, 8192 15.4 / 15.6 / 12.4; 4096 of 10 of 1000 12.9 / 11.3 / 10.4. A
// dispatch without items (two launches): 32768 assignments of 512 experts 10.5 / 11.5 / 10.0, 270000 24.5 / 42.5 / 22.4, of 1024 34.9 / 66 / 33.5.
constexpr int kWideExperts = kDispatchWide, kWideWaves = kChunk / 64;

__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) void dispatch_place_wide_k(
        const int * __restrict__ ids, const int * __restrict__ chunk_counts, int * __restrict__ counts, int * __restrict__ offsets, int * __restrict__ perm,
        int * __restrict__ groups, int capacity, int A, int E, int chunks, DispatchSide side) {
    extern __shared__ int hist[];   // kWideWaves x E: group sizes, then each wave's first place
    __shared__ int s_start[kWideExperts], s_all[kWideExperts], s_wave[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), chunk = blockIdx.x;
    const bool apart = chunk == chunks, plans = apart || (chunk == 0 && int(gridDim.x) == chunks);   // no chunk of its own; writes counts and plan
    const int a = chunk * kChunk + tid;
    int e = a < A ? ids[a] : -1;
    if (e >= E) e = -1;
    int before = 0, all = 0;
    const int * cc = chunk_counts;
    auto add_up = [&](auto together, auto whole, int b0) {   // so many loads in flight: the sums are latency, not bandwidth
        constexpr int N = decltype(together)::value;
        int v[N];
        const int * row = cc;
#pragma unroll
        for (int q = 0; q < N; ++q) {
            v[q] = decltype(whole)::value || b0 + q < chunks ? row[tid] : 0;
            row += E;                  // (q * E instead: sixteen lane addresses kept over the trips, 26 registers more)
        }
#pragma unroll
        for (int q = 0; q < N; ++q) { all += v[q]; before += b0 + q < chunk ? v[q] : 0; }
    };
    if (tid < E) {
        int b0 = 0;
#pragma unroll 1
        for (; chunks - b0 > 16; b0 += 16, cc += 16 * E) add_up(std::integral_constant<int, 16>{}, std::true_type{}, b0);
        if (chunks - b0 <= 8) add_up(std::integral_constant<int, 8>{}, std::false_type{}, b0);
        else add_up(std::integral_constant<int, 16>{}, std::false_type{}, b0);
    }
    if (!apart)
        for (int j = tid; j < kWideWaves * E; j += 1024) hist[j] = 0;
    // the experts' first places: a prefix sum over the threads
    const int incl = wave_scan(all);
    if (lane == 63) s_wave[wave] = incl;
    // the lanes of this wave with the same expert
    unsigned long long same = __ballot(e >= 0);
    for (int bit = 0; (1 << bit) < E; ++bit) {
        const unsigned long long m = __ballot((e >> bit) & 1);
        same &= ((e >> bit) & 1) ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull)), size = __popcll(same);
    __syncthreads();
    const int waves = row_scan(s_wave[lane & 15]), start = incl - all + (wave ? __builtin_amdgcn_readlane(waves, wave - 1) : 0);
    if (tid < E) { s_start[tid] = start; s_all[tid] = all; }
    if (!apart && e >= 0 && rank == size - 1) hist[wave * E + e] = size;
    __syncthreads();
    if (!apart) {
        if (tid < E) {
            int v[kWideWaves], at = start + before;
#pragma unroll
            for (int w = 0; w < kWideWaves; ++w) v[w] = hist[w * E + tid];
#pragma unroll
            for (int w = 0; w < kWideWaves; ++w) { hist[w * E + tid] = at; at += v[w]; }
        }
        __syncthreads();
        if (e >= 0) {
            const int place = hist[wave * E + e] + rank, slot = place - s_start[e];
            if (perm) perm[place] = a;
            if (groups && slot < capacity) groups[int64_t(e) * capacity + slot] = a;
        }
    }
    if (!plans) return;
    if (tid < E) { counts[tid] = all; if (offsets) offsets[tid] = start; }
    if (tid == E - 1 && offsets) offsets[E] = start + all;
    if (side.item_rows) plan_items(s_all, s_start, E, side.item_rows, side.items, side.index);
}

// A <= kChunk: everything in one block
__global__ __launch_bounds__(256) void dispatch_small_k(const int * __restrict__ ids, int * __restrict__ counts, int * __restrict__ offsets,
                                                        int * __restrict__ perm, int * __restrict__ groups, int capacity, int A, int E) {
    extern __shared__ int sm[];  // hist E, offs E + 1, scratch 256
    int * hist = sm, * offs = sm + E, * scratch = sm + 2 * E + 1;
    zero_lds(hist, E);
    __syncthreads();
    for (int a = threadIdx.x; a < A; a += 256) { const int e = ids[a]; if (e >= 0 && e < E) atomicAdd(&hist[e], 1); }
    __syncthreads();
    block_exclusive_scan(hist, offs, E, scratch);
    for (int j = threadIdx.x; j < E; j += 256) { counts[j] = hist[j]; if (offsets) offsets[j] = offs[j]; }
    if (threadIdx.x == 0 && offsets) offsets[E] = offs[E];
    __syncthreads();
    zero_lds(hist, E);
    __syncthreads();
    place_chunk(ids, offs, nullptr, perm, groups, capacity, 0, A, E, hist);
}

}  // namespace
}  // namespace tqmoe

using namespace tqmoe;

extern "C" uint32_t tqmoe_abi_version(void) { return TQMOE_ABI_VERSION; }

extern "C" int32_t tqmoe_router(const void * router, uint32_t wtype, const void * shared_gate, const void * x, uint32_t xtype,
                                float * logits, int32_t hidden, int32_t experts, int32_t n, void * stream, tqmoe_error * err) {
    if (!router || !x || !logits || hidden <= 0 || experts <= 0 || n <= 0) return fail(err, TQMOE_E_ARG, "tqmoe_router: invalid shape or pointer");
    if (hidden % 8) return fail(err, TQMOE_E_ARG, "tqmoe_router: hidden must be a multiple of 8");
    if ((wtype != TQMOE_F32 && wtype != TQMOE_BF16) || !is_act_type(xtype)) return fail(err, TQMOE_E_UNSUPPORTED, "tqmoe_router: unsupported element type");
    if ((n + kRouterTok - 1) / kRouterTok > 65535) return fail(err, TQMOE_E_ARG, "tqmoe_router: too many tokens for one call");
    if (int32_t rc = need_device(err, "tqmoe_router")) return rc;
    return enqueue_router(router, wtype, shared_gate, x, xtype, logits, hidden, experts, n, RouterSide{}, static_cast<hipStream_t>(stream), err);
}

int32_t tqmoe::enqueue_router(const void * router, uint32_t wtype, const void * shared_gate, const void * x, uint32_t xtype, float * logits, int hidden, int experts, int n,
                              const RouterSide & side, hipStream_t s, tqmoe_error * err) {
    if (wtype == xtype && (wtype == TQMOE_BF16 || wtype == TQMOE_F32) && int64_t(n) * (experts + 1) >= (wtype == TQMOE_F32 ? kRouterGemmMin<true> : kRouterGemmMin<false>) && hidden % 64 == 0 && !side.image) {
        if (wtype == TQMOE_F32) launch_router_gemm<true>(router, shared_gate, x, logits, hidden, experts, n, side, s);
        else launch_router_gemm<false>(router, shared_gate, x, logits, hidden, experts, n, side, s);
    } else if (wtype == TQMOE_F32) launch_router_x<TQMOE_F32>(xtype, router, shared_gate, x, logits, hidden, experts, n, side, s);
    else launch_router_x<TQMOE_BF16>(xtype, router, shared_gate, x, logits, hidden, experts, n, side, s);
    return launched(err, "tqmoe_router");
}

// top-k with the optional extras of the whole-layer path: extended ids and the input rows' activation image
namespace tqmoe {
int32_t enqueue_topk(const float * logits, int32_t * ids, float * weights, float * shared_weights, int32_t * ext_ids, int32_t extra, int32_t experts, int32_t topk, int32_t n,
                     float scale, int32_t gating, const float * bias, int32_t norm, int32_t shared_ungated, const TopkSide & side, hipStream_t s) {
    const TopkOut o{ids, weights, shared_weights, ext_ids, extra, shared_ungated, side};
    const uint32_t xt = side.rows ? side.xtype : uint32_t(TQMOE_F32);
    if (gating == TQMOE_GATE_SOFTMAX && !bias && norm) {   // the common case has its own kernel
        switch (xt) {
            case TQMOE_F32: launch_topk<TQMOE_F32>(logits, o, experts, topk, n, scale, s); break;
            case TQMOE_F16: launch_topk<TQMOE_F16>(logits, o, experts, topk, n, scale, s); break;
            default: launch_topk<TQMOE_BF16>(logits, o, experts, topk, n, scale, s); break;
        }
        return 0;
    }
    const Gate g{bias, gating, norm};
    switch (xt) {
        case TQMOE_F32: launch_topk_gated<TQMOE_F32>(logits, o, g, experts, topk, n, scale, s); break;
        case TQMOE_F16: launch_topk_gated<TQMOE_F16>(logits, o, g, experts, topk, n, scale, s); break;
        default: launch_topk_gated<TQMOE_BF16>(logits, o, g, experts, topk, n, scale, s); break;
    }
    return 0;
}
}  // namespace tqmoe

extern "C" int32_t tqmoe_topk(const float * logits, int32_t * ids, float * weights, float * shared_weights, int32_t experts,
                              int32_t topk, int32_t n, float scale, void * stream, tqmoe_error * err) {
    if (!logits || !ids || !weights || experts <= 0 || experts > 4096 || topk <= 0 || topk > experts || n <= 0)
        return fail(err, TQMOE_E_ARG, "tqmoe_topk: invalid shape or pointer");
    if (int32_t rc = need_device(err, "tqmoe_topk")) return rc;
    enqueue_topk(logits, ids, weights, shared_weights, nullptr, 0, experts, topk, n, scale, TQMOE_GATE_SOFTMAX, nullptr, 1, 0, TopkSide{}, static_cast<hipStream_t>(stream));
    return launched(err, "tqmoe_topk");
}

// The reference's moe_topk2 (src/experts/moe_kernels.cuh:24-25, src/experts/moe.cu:261-263): moe_topk on two routings in
// one launch, at most 1024 experts.
extern "C" int32_t tqmoe_topk2(const float * logits, int32_t * ids, float * weights, float * shared_weights, const float * logits2, int32_t * ids2,
                               float * weights2, float * shared_weights2, int32_t experts, int32_t topk, int32_t n, float scale, void * stream,
                               tqmoe_error * err) {
    if (!logits || !ids || !weights || !logits2 || !ids2 || !weights2 || experts <= 0 || experts > 1024 || topk <= 0 || topk > experts || n <= 0)
        return fail(err, TQMOE_E_ARG, "tqmoe_topk2: invalid shape or pointer (at most 1024 experts)");
    if (int32_t rc = need_device(err, "tqmoe_topk2")) return rc;
    const TopkOut o{ids, weights, shared_weights, nullptr, 0, 0, TopkSide{}}, o2{ids2, weights2, shared_weights2, nullptr, 0, 0, TopkSide{}};
    const dim3 grid(unsigned(n), 2);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (experts <= 64) topk2_reg_k<1><<<grid, 64, 0, s>>>(logits, o, logits2, o2, experts, topk, scale);
    else if (experts <= 128) topk2_reg_k<2><<<grid, 64, 0, s>>>(logits, o, logits2, o2, experts, topk, scale);
    else if (experts <= 256) topk2_reg_k<4><<<grid, 64, 0, s>>>(logits, o, logits2, o2, experts, topk, scale);
    else if (experts <= 512) topk2_reg_k<8><<<grid, 64, 0, s>>>(logits, o, logits2, o2, experts, topk, scale);
    else topk2_reg_k<16><<<grid, 64, 0, s>>>(logits, o, logits2, o2, experts, topk, scale);
    return launched(err, "tqmoe_topk2");
}

extern "C" int32_t tqmoe_topk_gated(const float * logits, const float * probs_bias, int32_t gating, int32_t norm_weights, int32_t * ids, float * weights,
                                    float * shared_weights, int32_t experts, int32_t topk, int32_t n, float scale, void * stream, tqmoe_error * err) {
    if (!logits || !ids || !weights || experts <= 0 || experts > 4096 || topk <= 0 || topk > experts || n <= 0)
        return fail(err, TQMOE_E_ARG, "tqmoe_topk_gated: invalid shape or pointer");
    if (gating < TQMOE_GATE_SOFTMAX || gating > TQMOE_GATE_SQRT_SOFTPLUS) return fail(err, TQMOE_E_UNSUPPORTED, "tqmoe_topk_gated: unsupported gating function %d", gating);
    if (int32_t rc = need_device(err, "tqmoe_topk_gated")) return rc;
    enqueue_topk(logits, ids, weights, shared_weights, nullptr, 0, experts, topk, n, scale, gating, probs_bias, norm_weights != 0, 0, TopkSide{},
                 static_cast<hipStream_t>(stream));
    return launched(err, "tqmoe_topk_gated");
}

extern "C" size_t tqmoe_dispatch_workspace_bytes(int32_t experts, int32_t n, int32_t topk) {
    if (experts <= 0 || n <= 0 || topk <= 0) return 0;
    const int64_t A = int64_t(n) * topk, chunks = (A + kChunk - 1) / kChunk;
    return chunks <= 1 ? 16 : size_t(chunks) * size_t(experts) * sizeof(int);
}

// Scratch of tqmoe_dispatch_static: the per-chunk counts (and, for a caller that passes no offsets array, the offsets the
// placement of more than 1024 experts reads), in the library's own device image (every GPU the library runs on holds its
// copy until the process ends). In host code the array's name is not a device address: the address on the current device
// comes from hipGetSymbolAddress, once per device, and only that pointer is handed to the kernels.
constexpr int kStaticInts = 1 << 20;                 // 4 MiB: chunks x experts may not exceed it
constexpr int kStaticOffsets = 4352;                 // behind them: room for the offsets of up to 4096 experts
static __device__ __align__(256) int scratch[kStaticInts + kStaticOffsets];

namespace tqmoe {
namespace {
void place_wide(const int32_t * ids, const int * cc, int32_t * counts, int32_t * offsets, int32_t * perm, int32_t * groups, int32_t capacity, int32_t experts, int A,
                int chunks, const DispatchSide & side, hipStream_t s) {
    allow_dynamic_lds(reinterpret_cast<const void *>(&dispatch_place_wide_k), int(kWideWaves * kWideExperts * sizeof(int)));
    const unsigned blocks = unsigned(chunks) + (side.item_rows && chunks < 256 ? 1 : 0);   // (one more than the compute units would open a second round)
    dispatch_place_wide_k<<<blocks, 1024, size_t(kWideWaves) * experts * sizeof(int), s>>>(ids, cc, counts, offsets, perm, groups, capacity, A, experts, chunks, side);
}
// the launches of tqmoe_dispatch; cc: chunks x experts ints of scratch for more than one chunk. offsets and perm may be
// null where the caller only wants counts and groups (spare_offsets: experts + 1 ints the scan may use instead).
int32_t enqueue_dispatch(const int32_t * ids, int32_t * counts, int32_t * offsets, int32_t * perm, int32_t * groups, int32_t capacity, int32_t experts,
                         int A, int chunks, int * cc, int * spare_offsets, hipStream_t s, tqmoe_error * err, const char * what) {
    if (chunks == 1) {
        dispatch_small_k<<<1, 256, size_t(2 * experts + 1 + 256) * sizeof(int), s>>>(ids, counts, offsets, perm, groups, capacity, A, experts);
        return launched(err, what);
    }
    dispatch_count_k<<<unsigned(chunks), 256, size_t(experts) * sizeof(int), s>>>(ids, cc, A, experts);
    if (experts <= kWideExperts) {
        place_wide(ids, cc, counts, offsets, perm, groups, capacity, experts, A, chunks, DispatchSide{}, s);
        return launched(err, what);
    }
    int32_t * offs = offsets ? offsets : spare_offsets;
    dispatch_scan_k<<<1, 1024, size_t(experts + 1024) * sizeof(int), s>>>(cc, counts, offs, chunks, experts);
    dispatch_place_k<<<unsigned(chunks), 256, size_t(experts) * sizeof(int), s>>>(ids, offs, cc, perm, groups, capacity, A, experts);
    return launched(err, what);
}

// Address of ::scratch on each device: looked up once (under the mutex), read without a lock afterwards.
constexpr int kMaxDevices = 64;
std::atomic<int *> g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mutex;

int32_t static_scratch(int ** out, tqmoe_error * err) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(err, TQMOE_E_DEVICE, "tqmoe_dispatch_static: no usable current device");
    int * p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
        if (!p) {
            void * sym = nullptr;
            const hipError_t rc = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch));
            if (rc != hipSuccess || !sym) return fail(err, TQMOE_E_DEVICE, "tqmoe_dispatch_static: hipGetSymbolAddress: %s", hipGetErrorString(rc));
            p = static_cast<int *>(sym);
            g_scratch_ptr[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    return 0;
}

// counts[ids[i]] += 1 as 64-bit counters (a routing profile that runs on over many calls)
__global__ __launch_bounds__(256) void count_k(const int * __restrict__ ids, unsigned long long * __restrict__ counts, int count) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < count) { const int e = ids[i]; if (e >= 0) atomicAdd(counts + e, 1ull); }
}

// The decode grouping maps of one routed call, one block. Assignment a has slot s = slot_of[ids[a]] (-1 for a skipped id).
// The assignments of a slot, in ascending a, are cut into runs of kDedupCols; the run is a group, groups are numbered by
// their first assignment. Every thread walks the slots of the assignments before it (LDS broadcast reads), which gives its
// rank in its slot and the assignment that opened its run; a block-wide prefix over the opening flags numbers the groups.
constexpr int kDedupCols = 8, kDedupStride = 2 + 2 * kDedupCols;
__global__ __launch_bounds__(1024) void dedup_maps_k(const int * __restrict__ ids, const int * __restrict__ slot_of, int count, int topk,
                                                     int * __restrict__ slots, int * __restrict__ gu, int * __restrict__ dn, int groups) {
    __shared__ int s_slot[1024], s_group[1024], s_wave[16];
    const int a = threadIdx.x, lane = a & 63, wave = a >> 6;
    for (int i = a; i < groups * kDedupStride; i += 1024) { if (gu) gu[i] = -1; if (dn) dn[i] = -1; }
    int s = -1;
    if (a < count) { const int e = ids[a]; s = e >= 0 ? slot_of[e] : -1; if (slots) slots[a] = s; }
    s_slot[a] = a < count ? s : -1;
    __syncthreads();
    int rank = 0, total = 0, opener = a;
    if (s >= 0) {
        for (int b = 0; b < count; ++b) {
            if (s_slot[b] != s) continue;
            if (b < a) { if ((rank & (kDedupCols - 1)) == 0) opener = b; ++rank; }
            ++total;
        }
        if ((rank & (kDedupCols - 1)) == 0) opener = a;
    }
    const bool opens = s >= 0 && (rank & (kDedupCols - 1)) == 0;
    const unsigned long long m = __ballot(opens);
    if (lane == 0) s_wave[wave] = __popcll(m);
    __syncthreads();
    int g = __popcll(m & ((1ull << lane) - 1ull));
    for (int w = 0; w < wave; ++w) g += s_wave[w];
    s_group[a] = g;                 // meaningful where the thread opens a group
    __syncthreads();
    if (s < 0) return;
    const int col = rank & (kDedupCols - 1), first = rank - col;
    int * maps[2] = {gu, dn};
#pragma unroll
    for (int part = 0; part < 2; ++part) {
        int * e = maps[part];
        if (!e) continue;
        e += int64_t(s_group[opener]) * kDedupStride;
        if (col == 0) { e[0] = s; e[1] = min(kDedupCols, total - first); }
        e[2 + col] = part ? a : a / topk;
        e[2 + kDedupCols + col] = a;
    }
}
}  // namespace

int32_t enqueue_layer_dispatch(const int32_t * ids, int32_t * counts, int32_t * offsets, int32_t * perm, int32_t experts, int32_t n, int32_t topk, int * chunk_counts,
                               const DispatchSide & side, hipStream_t s, tqmoe_error * err) {
    const int A = n * topk, chunks = (A + kChunk - 1) / kChunk;
    if (experts <= kWideExperts && (side.counted || chunks > 1)) {
        if (!side.counted) dispatch_count_k<<<unsigned(chunks), 256, size_t(experts) * sizeof(int), s>>>(ids, chunk_counts, A, experts);
        place_wide(ids, chunk_counts, counts, offsets, perm, nullptr, 0, experts, A, chunks, side, s);
        return launched(err, "tqmoe_layer_forward (dispatch)");
    }
    if (int32_t rc = enqueue_dispatch(ids, counts, offsets, perm, nullptr, 0, experts, A, chunks, chunk_counts, nullptr, s, err, "tqmoe_layer_forward (dispatch)")) return rc;
    if (side.item_rows) enqueue_grouped_plan(counts, offsets, experts, side.item_rows, side.items, side.index, s);
    return launched(err, "tqmoe_layer_forward (plan)");
}
}  // namespace tqmoe

extern "C" int32_t tqmoe_dispatch(const int32_t * ids, int32_t * counts, int32_t * offsets, int32_t * perm, int32_t * groups,
                                  int32_t capacity, int32_t experts, int32_t n, int32_t topk, void * workspace, size_t workspace_bytes,
                                  void * stream, tqmoe_error * err) {
    if (!ids || !counts || !offsets || !perm || experts <= 0 || experts > 4096 || n <= 0 || topk <= 0 || (groups && capacity <= 0))
        return fail(err, TQMOE_E_ARG, "tqmoe_dispatch: invalid shape or pointer");
    const int64_t A64 = int64_t(n) * topk;
    if (A64 > (1 << 30)) return fail(err, TQMOE_E_ARG, "tqmoe_dispatch: too many assignments");
    const int A = int(A64), chunks = (A + kChunk - 1) / kChunk;
    if (int32_t rc = need_device(err, "tqmoe_dispatch")) return rc;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (chunks > 1 && (!workspace || workspace_bytes < tqmoe_dispatch_workspace_bytes(experts, n, topk)))
        return fail(err, TQMOE_E_WORKSPACE, "tqmoe_dispatch: workspace of %zu bytes needed", tqmoe_dispatch_workspace_bytes(experts, n, topk));
    return enqueue_dispatch(ids, counts, offsets, perm, groups, capacity, experts, A, chunks, static_cast<int *>(workspace), nullptr, s, err, "tqmoe_dispatch");
}

extern "C" int32_t tqmoe_dispatch_static(const int32_t * ids, int32_t * counts, int32_t * offsets, int32_t * perm, int32_t * groups,
                                         int32_t capacity, int32_t experts, int32_t n, int32_t topk, void * stream, tqmoe_error * err) {
    if (!ids || !counts || experts <= 0 || experts > 4096 || n <= 0 || topk <= 0 || (groups && capacity <= 0) || (!groups && !perm))
        return fail(err, TQMOE_E_ARG, "tqmoe_dispatch_static: invalid shape or pointer");
    const int64_t A64 = int64_t(n) * topk, chunks64 = (A64 + kChunk - 1) / kChunk;
    if (A64 > (1 << 30)) return fail(err, TQMOE_E_ARG, "tqmoe_dispatch_static: too many assignments");
    if (chunks64 > 1 && chunks64 * experts > kStaticInts)
        return fail(err, TQMOE_E_WORKSPACE, "tqmoe_dispatch_static: %lld assignments x %d experts need %lld scratch ints, the built-in scratch holds %d "
                    "(use tqmoe_dispatch with a workspace)", (long long)A64, experts, (long long)(chunks64 * experts), kStaticInts);
    int * cc = nullptr;
    if (int32_t rc = static_scratch(&cc, err)) return rc;
    return enqueue_dispatch(ids, counts, offsets, perm, groups, capacity, experts, int(A64), int(chunks64), cc, cc + kStaticInts,
                            static_cast<hipStream_t>(stream), err, "tqmoe_dispatch_static");
}

extern "C" int32_t tqmoe_static_scratch_init(tqmoe_error * err) {
    int * p = nullptr;
    if (int32_t rc = need_device(err, "tqmoe_static_scratch_init")) return rc;
    return static_scratch(&p, err) ? TQMOE_E_DEVICE : ok(err);
}

extern "C" int32_t tqmoe_count(const int32_t * ids, uint64_t * counts, int32_t count, void * stream, tqmoe_error * err) {
    if (!ids || !counts || count <= 0) return fail(err, TQMOE_E_ARG, "tqmoe_count: invalid size or pointer");
    if (int32_t rc = need_device(err, "tqmoe_count")) return rc;
    count_k<<<unsigned((count + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(ids, reinterpret_cast<unsigned long long *>(counts), count);
    return launched(err, "tqmoe_count");
}

extern "C" int32_t tqmoe_dedup_maps(const int32_t * ids, const int32_t * slot_of, int32_t count, int32_t topk, int32_t * slots, int32_t * gu, int32_t * dn,
                                    int32_t groups, void * stream, tqmoe_error * err) {
    if (!ids || !slot_of || count <= 0 || count > 1024 || topk <= 0 || groups < count) return fail(err, TQMOE_E_ARG, "tqmoe_dedup_maps: invalid shape");
    if (int32_t rc = need_device(err, "tqmoe_dedup_maps")) return rc;
    dedup_maps_k<<<1, 1024, 0, static_cast<hipStream_t>(stream)>>>(ids, slot_of, count, topk, slots, gu, dn, groups);
    return launched(err, "tqmoe_dedup_maps");
}
