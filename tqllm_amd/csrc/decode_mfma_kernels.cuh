// Decode-sized products of the tile-major bank formats (IQ4_XS, Q4_K, Q6_K, IQ3_S, NVFP4G) on the matrix pipe.
//
// A block owns one expert, up to kTP of the input rows routed to it, and `tpw` tiles of 32 weight rows. Each wave takes
// one row tile and a share of the row's 256-weight super-blocks. Per 32-weight sub-block a lane (n = lane % 32,
// g = lane / 32) turns its half of weight row n's codes into 16 int8 values (MfmaFormat<FMT>::decode); that is operand
// B of v_mfma_i32_32x32x32_i8 (of two v_mfma_i32_32x32x16_i8 where the format has a scale per 16 weights). Operand A is
// the activation image: MFMA row 2j is the hi plane and row 2j + 1 the lo
// plane of input row j (rows past 2 kTP repeat others), read straight from the image because its plane order is the order B's
// bytes come in. The MFMA does the 32-term sums for all rows and planes at once, so no lane exchange is needed; its
// result registers 0..3 of lane half g are (hi, lo) of input rows 2g and 2g + 1, which one fp32 multiply-add each folds
// into the lane's running sum with weight scale * activation scale. Waves that split a row's super-blocks add their
// partial sums through LDS in wave order (deterministic).
// The weight bytes are the only cold data: every wave loads its share (codes and scale records) into registers one
// super-block ahead of the one it is multiplying, so the loads of the next super-block are in flight while this one is
// decoded.
//
// Why not v_dot4 products with a lane per sub-block (what the row-major formats run): those multiply every decoded weight
// with both planes of every input row in the vector pipe (16 instructions per 32 weights and row) and serve two rows a
// block; here the vector pipe only decodes and applies four scales per sub-block, and a block serves four rows.
#pragma once
#include "act_image.cuh"
#include "decode_chunks.cuh"
#include "decode_api.cuh"
#include "decode_table.cuh"
#include "formats.cuh"
#include "topk_select.cuh"

namespace tqmoe {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kTP = kChunkRowsMax;   // input rows per block
constexpr int kMaxWaves = 8;
constexpr int kStagedFrom = 12;      // assignments from which a block's input rows go through LDS (see mfma_launch)

constexpr int kIq4Table[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
constexpr int kFp4Table[16] = {0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12};   // twice the E2M1 values
__device__ __forceinline__ v4i decode_table(const Table16 & t, uint2 c) {
    const uint32_t m = 0x0F0F0F0Fu;
    return v4i{int(pick(t, c.x & m)), int(pick(t, (c.x >> 4) & m)), int(pick(t, c.y & m)), int(pick(t, (c.y >> 4) & m))};
}

// Every other sub-block (down_combine_k with half tiles): half_codes loads sub-blocks odd, odd + 2, ... into the places of 0, 2, ...;
// odd_rec moves their scales (minimums, index bits) there; d and dmin are read from the record as it was.
// What the kernel needs of a format. A lane's part of a super-block: Codes and Rec, loaded from the tile's code and record
// blocks (kCodeBytes, kRecBytes per tile and super-block). decode: operand B of sub-block ib. Scales: kGroups integer
// scales per sub-block (kFloat: fp32 ones) with the super-block's d behind them; kMin: a minimum per sub-block times the
// activations' sum. row_factor: a factor of the whole weight row.
template <uint32_t FMT> struct MfmaFormat;
struct MfmaBase {
    static constexpr int kGroups = 1;
    static constexpr bool kFloat = false, kMin = false, kRowFactor = false;
    static constexpr int kLattice = 1;
    static __device__ __forceinline__ float row_factor(const BankView &, int64_t) { return 1.f; }
};
struct MfmaNibbles : MfmaBase {   // sixteen code bytes a sub-block in the canonical order
    static constexpr int kCodeBytes = 4096;
    struct Codes { uint2 c[8]; };
    static __device__ __forceinline__ void codes(const uint8_t * p, int n, int g, Codes & c) {
        const uint8_t * q = p + n * 16 + g * 8;
#pragma unroll
        for (int ib = 0; ib < 8; ++ib) c.c[ib] = *reinterpret_cast<const uint2 *>(q + ib * 512);
    }
    static __device__ __forceinline__ void half_codes(const uint8_t * p, int n, int g, int odd, Codes & c) {
        const uint8_t * q = p + n * 16 + g * 8 + odd * 512;
#pragma unroll
        for (int ib = 0; ib < 8; ib += 2) c.c[ib] = *reinterpret_cast<const uint2 *>(q + ib * 512);
    }
};
template <> struct MfmaFormat<TQMOE_IQ4_XS> : MfmaNibbles {
    static constexpr int kRecBytes = 256;
    typedef uint2 Rec;
    static __device__ __forceinline__ Rec rec(const uint8_t * p, int n) { return *reinterpret_cast<const uint2 *>(p + n * 8); }
    static __device__ __forceinline__ v4i decode(const Codes & c, const Rec &, int ib, int, const uint32_t *) {
        constexpr Table16 t = table16(kIq4Table);
        return decode_table(t, c.c[ib]);
    }
    static __device__ __forceinline__ int scale(const Rec & r, int ib, int) { return iq4xs_lsm32(r, ib); }
    static __device__ __forceinline__ float d(const Rec & r) { return half_bits_to_float(iq4xs_d_bits(r)); }
    static __device__ __forceinline__ Rec odd_rec(const Rec & r, int odd) {   // five fields in x, then three from bit 14 of y: the fifth's successor is y's first
        return make_uint2(odd ? ((r.x >> 6) & 0x00FFFFFFu) | ((r.y << 10) & 0x3F000000u) : r.x, r.y >> (6 * odd));
    }
};
template <> struct MfmaFormat<TQMOE_Q4_K> : MfmaNibbles {
    static constexpr int kRecBytes = 512;
    static constexpr bool kMin = true;
    typedef uint4 Rec;
    static __device__ __forceinline__ Rec rec(const uint8_t * p, int n) { return *reinterpret_cast<const uint4 *>(p + n * 16); }
    static __device__ __forceinline__ v4i decode(const Codes & c, const Rec &, int ib, int, const uint32_t *) {
        const uint32_t m = 0x0F0F0F0Fu;
        return v4i{int(c.c[ib].x & m), int((c.c[ib].x >> 4) & m), int(c.c[ib].y & m), int((c.c[ib].y >> 4) & m)};
    }
    static __device__ __forceinline__ int scale(const Rec & r, int ib, int) {
        const uint32_t q[3] = {r.y, r.z, r.w};
        int sc, mn;
        q4k_scale_min(q, ib, sc, mn);
        return sc;
    }
    static __device__ __forceinline__ float minimum(const Rec & r, int ib) {
        const uint32_t q[3] = {r.y, r.z, r.w};
        int sc, mn;
        q4k_scale_min(q, ib, sc, mn);
        return float(mn);
    }
    static __device__ __forceinline__ float d(const Rec & r) { return half_bits_to_float(uint16_t(r.x & 0xFFFFu)); }
    static __device__ __forceinline__ float dmin(const Rec & r) { return half_bits_to_float(uint16_t(r.x >> 16)); }
    static __device__ __forceinline__ Rec odd_rec(const Rec & r, int odd) { return make_uint4(r.x, r.y >> (8 * odd), r.z >> (8 * odd), r.w >> (8 * odd)); }
};
template <> struct MfmaFormat<TQMOE_NVFP4G> : MfmaNibbles {
    static constexpr int kRecBytes = 512, kGroups = 2;
    static constexpr bool kFloat = true, kRowFactor = true;
    typedef uint4 Rec;   // the sixteen scale bytes
    static __device__ __forceinline__ Rec rec(const uint8_t * p, int n) {
        const uint2 a = *reinterpret_cast<const uint2 *>(p + n * 8), b = *reinterpret_cast<const uint2 *>(p + 256 + n * 8);
        return make_uint4(a.x, a.y, b.x, b.y);
    }
    static __device__ __forceinline__ v4i decode(const Codes & c, const Rec &, int ib, int, const uint32_t *) {
        constexpr Table16 t = table16(kFp4Table);
        return decode_table(t, c.c[ib]);
    }
    static __device__ __forceinline__ float scale(const Rec & r, int ib, int grp) {
        const uint32_t w = ib < 2 ? r.x : ib < 4 ? r.y : ib < 6 ? r.z : r.w;
        switch (2 * (ib & 1) + grp) {
            case 0: return __builtin_amdgcn_cvt_f32_fp8(int(w), 0);
            case 1: return __builtin_amdgcn_cvt_f32_fp8(int(w), 1);
            case 2: return __builtin_amdgcn_cvt_f32_fp8(int(w), 2);
            default: return __builtin_amdgcn_cvt_f32_fp8(int(w), 3);
        }
    }
    static __device__ __forceinline__ float d(const Rec &) { return 1.f; }
    static __device__ __forceinline__ Rec odd_rec(const Rec & r, int odd) { return make_uint4(r.x >> (16 * odd), r.y >> (16 * odd), r.z >> (16 * odd), r.w >> (16 * odd)); }
    static __device__ __forceinline__ float row_factor(const BankView & b, int64_t row) {   // half the row's global: the table holds twice the values
        return 0.5f * *reinterpret_cast<const float *>(b.aux + nvfp4_global_offset(b.rows_total, b.cols) + row * 4);
    }
};
template <> struct MfmaFormat<TQMOE_IQ3_S> : MfmaBase {
    static constexpr int kCodeBytes = 3072, kRecBytes = 512, kLattice = 2304;
    struct Codes { uint2 qs[4]; uint4 sg[2]; };
    typedef uint4 Rec;
    static __device__ __forceinline__ void codes(const uint8_t * p, int n, int g, Codes & c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c.qs[i] = *reinterpret_cast<const uint2 *>(p + i * 512 + n * 16 + g * 8);
#pragma unroll
        for (int i = 0; i < 2; ++i) c.sg[i] = *reinterpret_cast<const uint4 *>(p + 2048 + i * 512 + n * 16);
    }
    static __device__ __forceinline__ Rec rec(const uint8_t * p, int n) { return *reinterpret_cast<const uint4 *>(p + n * 16); }
    // The lattice in LDS holds eight times the odd magnitudes: 8 (2 k + 1) is the byte k << 4 | 8, and its negative the same
    // byte with the upper four bits inverted, so that a sign is one exclusive or.
    // Points 0..255 are the first 1 KB; the others follow 1, 2, 4 and 8 KB behind it, so that an index's ninth bit q of the four at
    // a time is an address bit where it stands (and a sign bit is a selector where it stands: seven of 45 instructions a sub-block
    // less; 64 tokens, top-8 of 256: 163.9 -> 157.2 us a layer).
    static __device__ __forceinline__ void lattice(uint32_t * lat, int tid, int threads) {
        for (int i = tid; i < 512; i += threads) {
            const uint32_t m = d_iq3s_grid.v[i] << 3;
            if (i < 256) lat[i] = m;
            else for (int q = 0; q < 4; ++q) lat[(256 << q) + i - 256] = m;
        }
    }
    // lookup: the four points' magnitudes, on their way from LDS; signed_of: with the signs
    static __device__ __forceinline__ v4i lookup(const Codes & c, const Rec & r, int ib, int g, const uint32_t * lat) {
        const uint32_t qs = (ib & 1) ? c.qs[ib >> 1].y : c.qs[ib >> 1].x;
        const uint32_t qh = (((ib < 4 ? r.y : r.z) >> (8 * (ib & 3))) >> (4 * g)) << 10;
        v4i w;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t low = ((qs >> (8 * q)) & 0xFFu) << 2;   // (a byte shifted: one instruction, where nothing is merged into it)
            asm("" : "+v"(low));
            w[q] = *reinterpret_cast<const int *>(reinterpret_cast<const uint8_t *>(lat) + (low | (qh & (0x400u << q))));
        }
        return w;
    }
    static __device__ __forceinline__ v4i signed_of(v4i w, const Codes & c, int ib, int g) {
        const uint4 s4 = c.sg[ib >> 2];
        const uint32_t sg = ((ib & 3) == 0 ? s4.x : (ib & 3) == 1 ? s4.y : (ib & 3) == 2 ? s4.z : s4.w) >> (4 * g);
        // A sign bit where it stands (a byte 0 or 1 << q) picks from a pool with 0x00 at 0 and 0xF0 at 1, 2 and 4; 8 picks the sign of
        // the pool's byte 1 in all bits.
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t m = __builtin_amdgcn_perm(0x000000F0u, 0x00F0F000u, sg & (0x01010101u << q));
            w[q] ^= int(q < 3 ? m : m & 0xF0F0F0F0u);
        }
        return w;
    }
    static __device__ __forceinline__ v4i decode(const Codes & c, const Rec & r, int ib, int g, const uint32_t * lat) { return signed_of(lookup(c, r, ib, g, lat), c, ib, g); }
    static __device__ __forceinline__ void half_codes(const uint8_t * p, int n, int g, int odd, Codes & c) {
        codes(p, n, g, c);
#pragma unroll
        for (int i = 0; i < 4; ++i) c.qs[i].x = odd ? c.qs[i].y : c.qs[i].x;
#pragma unroll
        for (int i = 0; i < 2; ++i) { c.sg[i].x = odd ? c.sg[i].y : c.sg[i].x; c.sg[i].z = odd ? c.sg[i].w : c.sg[i].z; }
    }
    static __device__ __forceinline__ Rec odd_rec(const Rec & r, int odd) { return make_uint4(r.x >> (4 * odd), r.y >> (8 * odd), r.z >> (8 * odd), r.w >> (4 * odd)); }
    static __device__ __forceinline__ int scale(const Rec & r, int ib, int) { return 1 + 2 * iq3s_ls(r, ib); }
    static __device__ __forceinline__ float d(const Rec & r) { return 0.125f * half_bits_to_float(uint16_t(r.x & 0xFFFFu)); }
};
template <> struct MfmaFormat<TQMOE_Q6_K> : MfmaBase {
    static constexpr int kCodeBytes = 6144, kRecBytes = 1024, kGroups = 2;
    struct Codes { uint2 lo[8]; uint2 hi[4]; };
    struct Rec { uint4 sc; uint32_t d; };
    static __device__ __forceinline__ void codes(const uint8_t * p, int n, int g, Codes & c) {
        const uint8_t * q = p + n * 16 + g * 8;
#pragma unroll
        for (int ib = 0; ib < 8; ++ib) c.lo[ib] = *reinterpret_cast<const uint2 *>(q + ib * 512);
#pragma unroll
        for (int i = 0; i < 4; ++i) c.hi[i] = *reinterpret_cast<const uint2 *>(q + 4096 + i * 512);
    }
    static __device__ __forceinline__ Rec rec(const uint8_t * p, int n) {
        return Rec{*reinterpret_cast<const uint4 *>(p + n * 32), *reinterpret_cast<const uint16_t *>(p + n * 32 + 16)};
    }
    static __device__ __forceinline__ v4i decode(const Codes & c, const Rec &, int ib, int, const uint32_t *) {
        uint32_t w[4];
        q6k_times4(c.lo[ib], (ib & 1) ? c.hi[ib >> 1].y : c.hi[ib >> 1].x, w);
        return v4i{int(w[0]), int(w[1]), int(w[2]), int(w[3])};
    }
    static __device__ __forceinline__ int scale(const Rec & r, int ib, int grp) {
        const uint32_t w = ib < 2 ? r.sc.x : ib < 4 ? r.sc.y : ib < 6 ? r.sc.z : r.sc.w;
        return __builtin_amdgcn_sbfe(int(w), 8 * (2 * (ib & 1) + grp), 8);
    }
    static __device__ __forceinline__ float d(const Rec & r) { return 0.25f * half_bits_to_float(uint16_t(r.d)); }
    static __device__ __forceinline__ void half_codes(const uint8_t * p, int n, int g, int odd, Codes & c) {
        const uint8_t * q = p + n * 16 + g * 8;
#pragma unroll
        for (int ib = 0; ib < 8; ib += 2) c.lo[ib] = *reinterpret_cast<const uint2 *>(q + (ib + odd) * 512);
#pragma unroll
        for (int i = 0; i < 4; ++i) c.hi[i].x = *reinterpret_cast<const uint32_t *>(q + 4096 + i * 512 + odd * 4);
    }
    static __device__ __forceinline__ Rec odd_rec(const Rec & r, int odd) {
        return Rec{make_uint4(r.sc.x >> (16 * odd), r.sc.y >> (16 * odd), r.sc.z >> (16 * odd), r.sc.w >> (16 * odd)), r.d};
    }
};

// NB banks (gate and up, or one). gateup != 0: out0 is the activation image that receives silu(gate) * up; else out0 /
// out1 receive the products as rows of `ytype`. wk waves share a row's super-blocks, tpw row tiles per block.
// Dynamic LDS: the partial sums and, behind them, the input rows' planes and scales (MODE 1, 2): nothing of the one lies in the other, so that a
// pass's sums need no barrier in front but where another pass (MODE 2) has left its own there.
// UNI: every sub-block of an input row has the row's one activation scale (the images tqmoe_quant_act and the top-k
// kernel write). The 6-bit weight scales then multiply the integer results and the sums stay integers over a whole
// super-block; otherwise (rows quantised block by block, as the fused gate / up epilogue leaves them) each sub-block's
// result is scaled in fp32.
// MODE 0: input rows read straight from the image; 1: staged in LDS; 2: staged, and a wave takes tl_count row tiles in turn
// Three waves a SIMD (168 registers) where that does not spill; two for the two-bank kernels of the formats with more codes or
// scales in registers.
// ROUTE (MODE 0): the block selects its own expert from the token's logits (up to 64 ROUTE experts); see DecodeTopk.
template <uint32_t FMT, int NB, bool UNI, int MODE>
constexpr int kDecodeWaves = NB == 2 && (FMT == TQMOE_Q6_K || (MODE == 0 && (FMT == TQMOE_Q4_K || (!UNI && FMT != TQMOE_IQ4_XS)))) ? 2 : 3;
template <uint32_t FMT, int NB, bool UNI, int MODE, int ROUTE = 0>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(kDecodeWaves<FMT, NB, UNI, MODE>))) void decode_mfma_k(BankView b0, BankView b1, const uint8_t * __restrict__ image, void * out0, void * out1, uint32_t ytype,
                                                    const int * __restrict__ ids, int A, int xdiv, int mode, int slots, int topk, int shared_lim, int wk,
                                                    int tpw, int gateup, int a_off, int tl_count, Glu glu, DecodeTopk route) {
    using F = MfmaFormat<FMT>;
    constexpr bool STAGED = MODE >= 1, MULTI = MODE == 2;
    constexpr int kIn = ROUTE > 0 ? 1 : 2;   // input rows a lane half has sums of (a block that routes serves one)
    extern __shared__ __attribute__((aligned(16))) uint8_t stage[];
    __shared__ int meta[1], s_tok[kTP];
    __shared__ float s_x0[kTP];
    __shared__ __attribute__((aligned(16))) int ql[kMaxWaves * 2][32];
    __shared__ uint32_t lat[F::kLattice];
    if constexpr (FMT == TQMOE_IQ3_S)   // eight times the magnitudes (behind a barrier before the first use)
        F::lattice(lat, threadIdx.x, blockDim.x);
    // ROUTE: blockIdx.y is the token, blockIdx.x the slot and its group of row tiles (behind a block that only writes the routing down)
    const int at = ROUTE > 0 ? int(blockIdx.x) - route.apart : 0, slot = ROUTE == 0 || at < 0 ? 0 : route.groups == 1 ? at : int(__umulhi(uint32_t(at), route.per_group));
    const int a = ROUTE > 0 ? int(blockIdx.y) * slots + slot : int(blockIdx.y), bx = ROUTE > 0 ? at - slot * route.groups : int(blockIdx.x);   // bx: the block's group of row tiles
    const int S = b0.cols / 32, NSB = S / 8, rows = b0.rows, tiles = rows / 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 31, g = lane >> 5;
    // ROUTE: the block's one input row is known before its expert is: the row's first operands and its scale are loaded, and everything
    // that does not depend on the expert is worked out, while that is selected (of 14600 cycles of the block 3700 passed before the
    // expert was known, 1200 in setting up behind it, and the operands' trip began after the weights'; eight layers of one
    // token over 512 experts 139 -> 128 us, four of 64 experts 63.9 -> 60)
    constexpr bool EARLY = ROUTE > 0 && FMT != TQMOE_NVFP4G;   // (NVFP4G's scales leave no registers for them)
    [[maybe_unused]] v4i a_row[EARLY ? 8 : 1];
    [[maybe_unused]] float4 m_row[2];
    [[maybe_unused]] float x_row = 0.f;
    const uint8_t * const row_a = ROUTE > 0 ? image_row_ptr(image, blockIdx.y, S) : nullptr;
    auto fetch_row = [&](int sb) {
        if constexpr (EARLY) {
#pragma unroll
            for (int i = 0; i < 8; ++i) a_row[i] = *reinterpret_cast<const v4i *>(row_a + (sb * 8 + i) * 64 + (n & 1) * 32 + g * 16);
            if constexpr (F::kMin) {
                m_row[0] = *reinterpret_cast<const float4 *>(image_sums(row_a, S) + sb * 8);
                m_row[1] = *reinterpret_cast<const float4 *>(image_sums(row_a, S) + sb * 8 + 4);
            }
        }
    };
    int e, wk_i, rt_l, n_tok = 1;
    int tok[kTP] = {a, -1, -1, -1};
    if constexpr (ROUTE > 0) {
        // One wave selects, for as many rounds as its assignment needs. The token's whole routing is written down by a block of its own,
        // so that the weights' exponentials and divisions are in nobody's way (one token of the 512-expert IQ4_XS layer, launch 10.0 ->
        // 9.3 us), or, where such blocks would open another round of the compute units, by the last slot's first block (4096 x 512 experts, top-4,
        // four tokens, 256 blocks: NVFP4G 25.5 us a layer so, 33 with blocks apart).
        const int token = blockIdx.y;
        const float * x = route.logits + int64_t(token) * (route.experts + 1);
        const bool writes = route.apart ? at < 0 : bx == 0 && slot == slots - 1;
        TopkLogits<ROUTE> logits;
        if (wave == 0) logits = topk_logits<ROUTE>(x, route.experts, lane);
        rt_l = (wave >= wk) + (wave >= 2 * wk) + (wave >= 3 * wk), wk_i = wave - rt_l * wk;
        fetch_row(wk_i);
        x_row = image_scales(row_a, S)[0];
        if (wave == 0 && (writes || slot < topk)) {
            const float shared_logit = writes && route.shared_weights ? x[route.experts] : 0.f;
            int my_id;
            float my_w;
            topk_select<ROUTE>(logits, route.experts, writes ? topk : slot + 1, lane, writes, &ql[0][0], my_id, my_w);
            if (lane == slot) meta[0] = my_id;
            if (writes) {
                const float v = topk_weight(my_w, topk, route.scale);
                if (lane < topk) { route.ids[int64_t(token) * topk + lane] = my_id; route.weights[int64_t(token) * topk + lane] = v; }
                if (lane == 0 && route.shared_weights) route.shared_weights[token] = route.shared_ungated ? 1.f : 1.f / (1.f + expf(-shared_logit));
            }
        }
        if (at < 0) return;
        __syncthreads();
        e = slot < topk ? meta[0] : route.experts;
    } else {
        n_tok = chunk_rows(ids, A, a, mode, e, tok);
        rt_l = (wave >= wk) + (wave >= 2 * wk) + (wave >= 3 * wk), wk_i = wave - rt_l * wk;   // (at most four row tiles: divisions were a tenth of a short launch's instructions)
    }
    if (e < 0 || int64_t(e) * b0.rows >= b0.rows_total) return;   // skipped assignment, or an id outside the bank
    if (n_tok == 0) return;
    if (ROUTE == 0 && threadIdx.x < kTP) s_tok[threadIdx.x] = tok[threadIdx.x];

    const int tile = bx * tl_count * tpw + rt_l;   // the wave's first (or only) row tile
    const bool shared_slot = ROUTE > 0 ? slot >= topk : (a % slots) >= topk;
    // the shared expert may have fewer rows (gate / up) or read a narrower input row (down)
    const int row_lim = gateup && shared_slot ? shared_lim : rows;
    const int s_end = !gateup && shared_slot ? shared_lim / 32 : S;
    const bool valid = tile < tiles && tile * 32 < row_lim;

    // The weight bytes of a super-block: 8 bytes of codes per sub-block and the row's scale record, per lane, in
    // registers. The next super-block's are loaded before this one is multiplied (into the other of two sets that swap
    // roles, no copies), so that there are always loads in flight under the decode work. Past the wave's last
    // super-block the same one is fetched again: a branch around the loads would make every wait a wait for all of them.
    // The first super-block's loads go out before the input rows are staged: the two trips to memory overlap.
    const int sb_end = s_end / 8;   // whole super-blocks only (the launcher checks)
    const bool working = valid && wk_i < sb_end;
    struct Cold { typename F::Codes code[NB]; typename F::Rec rec[NB]; };
    // the lane's addresses in the wave's first row tile, worked out once; a fetch adds 32-bit offsets (dt row tiles further on)
    const uint8_t * code_base[NB], * rec_base[NB];
    {
        const int64_t at = (int64_t(e) * tiles + tile) * NSB;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            code_base[nb] = (nb ? b1 : b0).codes + at * F::kCodeBytes;
            rec_base[nb] = (nb ? b1 : b0).aux + at * F::kRecBytes;
        }
    }
    auto fetch_tile = [&](int dt, int sb, Cold & c) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            F::codes(code_base[nb] + uint32_t(dt * NSB + sb) * uint32_t(F::kCodeBytes), n, g, c.code[nb]);
            c.rec[nb] = F::rec(rec_base[nb] + uint32_t(dt * NSB + sb) * uint32_t(F::kRecBytes), n);
        }
    };
    auto fetch = [&](int sb, Cold & c) { fetch_tile(0, sb, c); };
    Cold c0, c1;
    if (working) fetch(wk_i, c0);
    // The planes and scales of the block's input rows go to LDS once: [sub-block][input row][64 bytes of planes], then
    // [input row][sub-block] scales. The product loop then has no loads from memory but the weights', so that its waits
    // count exactly those (a wait for an operand A load would also wait for every weight load issued before it).
    uint8_t * a_lds = stage + a_off;
    float * xs_lds = reinterpret_cast<float *>(a_lds + S * 256);
    [[maybe_unused]] float * sum_lds = xs_lds + (UNI ? 0 : S * kTP);      // formats with minimums: the activations' sums
    if constexpr (STAGED) {
        const uint8_t * src_row[kTP];
#pragma unroll
        for (int j = 0; j < kTP; ++j) src_row[j] = image_row_ptr(image, (tok[j] >= 0 ? tok[j] : tok[0]) / xdiv, S);   // rows not served: the first row's
        for (int i0 = threadIdx.x; i0 < S * 16; i0 += 4 * blockDim.x) {   // four pieces a thread per trip to memory
            auto piece = [&](int q) {   // past the end: the last piece again, not stored
                const int i = min(i0 + q * int(blockDim.x), S * 16 - 1), j = (i >> 2) & 3;
                const uint8_t * row = j == 0 ? src_row[0] : j == 1 ? src_row[1] : j == 2 ? src_row[2] : src_row[3];
                return *reinterpret_cast<const uint4 *>(row + (i >> 4) * 64 + (i & 3) * 16);
            };
            auto put = [&](int q, const uint4 & v) {
                const int i = i0 + q * int(blockDim.x);
                if (i < S * 16) *reinterpret_cast<uint4 *>(a_lds + i * 16) = v;
            };
            // (four named values, not an array: an array indexed in two loops has been placed in scratch memory by the compiler,
            // one trip to memory per piece)
            const uint4 v0 = piece(0), v1 = piece(1), v2 = piece(2), v3 = piece(3);
            put(0, v0); put(1, v1); put(2, v2); put(3, v3);
        }
        if constexpr (UNI) {   // the rows' one scale each
            if (threadIdx.x < kTP) {
                const int j = threadIdx.x;
                s_x0[j] = image_scales(j == 0 ? src_row[0] : j == 1 ? src_row[1] : j == 2 ? src_row[2] : src_row[3], S)[0];
            }
        }
        if constexpr (!UNI || F::kMin)
            for (int i = threadIdx.x; i < S * kTP; i += blockDim.x) {
                const int j = i / S;
                const uint8_t * row = j == 0 ? src_row[0] : j == 1 ? src_row[1] : j == 2 ? src_row[2] : src_row[3];
                if constexpr (!UNI) xs_lds[i] = image_scales(row, S)[i - j * S];
                if constexpr (F::kMin) sum_lds[i] = image_sums(row, S)[i - j * S];
            }
    }
    if constexpr (ROUTE == 0) __syncthreads();

    float accf[NB][2], accm[NB][2];   // products; minimums times the activations' sums
    auto clear = [&]() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) accf[nb][0] = accf[nb][1] = accm[nb][0] = accm[nb][1] = 0.f;
    };
    clear();

    // A row tile's sums to their place. tile0: the block's first row tile of this pass.
    auto finish = [&](int tile0, bool wave_valid) {
        if constexpr (UNI) {
            if (wave_valid) {   // the rows' own scales, once
                const float x0 = ROUTE > 0 ? x_row : STAGED ? s_x0[2 * g] : image_scales(image_row_ptr(image, max(s_tok[2 * g], 0) / xdiv, S), S)[0];
                const float x1 = ROUTE > 0 ? 0.f : STAGED ? s_x0[2 * g + 1] : image_scales(image_row_ptr(image, max(s_tok[2 * g + 1], 0) / xdiv, S), S)[0];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) { accf[nb][0] *= x0; accf[nb][1] *= x1; }
            }
        }
        if constexpr (F::kMin) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) { accf[nb][0] -= accm[nb][0]; accf[nb][1] -= accm[nb][1]; }
        }
        if constexpr (F::kRowFactor) {
            if (wave_valid) {
                const int64_t row = int64_t(e) * rows + (tile0 + rt_l) * 32 + n;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) { const float f = F::row_factor(nb ? b1 : b0, row); accf[nb][0] *= f; accf[nb][1] *= f; }
            }
        }
        if constexpr (MULTI) __syncthreads();                  // the previous pass's sums are done with
        float (*red)[NB][kTP][32] = reinterpret_cast<float (*)[NB][kTP][32]>(stage);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) { red[wave][nb][2 * g][n] = accf[nb][0]; red[wave][nb][2 * g + 1][n] = accf[nb][1]; }
        __syncthreads();

        // the waves of a row tile hold the partial sums of its super-block shares: added here in wave order
        const int groups = tpw * kTP, per_pass = blockDim.x >> 5;
        for (int g0 = 0; g0 < groups; g0 += per_pass) {   // every wave runs every pass: the image quantiser exchanges lanes
            const int grp = g0 + (threadIdx.x >> 5), i = threadIdx.x & 31;
            const int rt = grp / kTP, j = grp % kTP, t = tile0 + rt;
            const bool live = grp < groups && j < n_tok && t < tiles && t * 32 < row_lim;
            float v0 = 0.f, v1 = 0.f;
            if (live)
                for (int w = 0; w < wk; ++w) { v0 += red[rt * wk + w][0][j][i]; if (NB == 2) v1 += red[rt * wk + w][NB - 1][j][i]; }
            const int aj = ROUTE > 0 ? a : live ? s_tok[j] : 0;
            if (gateup) {
                glu_clamp_inputs(glu, v0, v1);
                const float act = glu_clamp_silu(glu, v0 / (1.f + expf(-v0))) * v1;
                quantise_block_lanes(act, i, live, ql[threadIdx.x >> 5], static_cast<uint8_t *>(out0) + int64_t(aj) * tiles * kImageSubBytes, tiles, t);
            } else if (live) {
                const int64_t o = int64_t(aj) * rows + t * 32 + i;
                if (ytype == TQMOE_F32) { static_cast<float *>(out0)[o] = v0; if (NB == 2) static_cast<float *>(out1)[o] = v1; }
                else { static_cast<uint16_t *>(out0)[o] = float_to_bf16_bits(v0); if (NB == 2) static_cast<uint16_t *>(out1)[o] = float_to_bf16_bits(v1); }
            }
        }
    };

    if (working) {
        // this lane's part of operand A: plane row n of the MFMA = plane (n & 1) of input row n >> 1 (rows 8 and up repeat
        // rows 0..7: their sums land in result rows that nobody reads)
        // (not staged: straight from the image, a stride of 64 bytes per sub-block instead of the staged 256)
        const uint8_t * a_lane = ROUTE > 0 ? row_a + (n & 1) * 32 + g * 16 : STAGED ? a_lds + ((n & 7) >> 1) * 64 + (n & 1) * 32 + g * 16
                                                : image_row_ptr(image, max(s_tok[(n & 7) >> 1], s_tok[0]) / xdiv, S) + (n & 1) * 32 + g * 16;
        constexpr int kStrideA = STAGED ? 256 : 64;
        // the two input rows whose sums land in this lane half's result registers
        const float * sc0 = ROUTE > 0 ? nullptr : STAGED ? xs_lds + (2 * g) * S : image_scales(image_row_ptr(image, max(s_tok[2 * g], 0) / xdiv, S), S);
        const float * sc1 = ROUTE > 0 ? nullptr : STAGED ? xs_lds + (2 * g + 1) * S : image_scales(image_row_ptr(image, max(s_tok[2 * g + 1], 0) / xdiv, S), S);
        const float * sum0 = ROUTE > 0 ? image_sums(row_a, S) : STAGED ? sum_lds + (2 * g) * S : image_sums(image_row_ptr(image, max(s_tok[2 * g], 0) / xdiv, S), S);
        const float * sum1 = ROUTE > 0 ? nullptr : STAGED ? sum_lds + (2 * g + 1) * S : image_sums(image_row_ptr(image, max(s_tok[2 * g + 1], 0) / xdiv, S), S);
        auto multiply = [&](int sb, const Cold & cur) {
            // Staged rows: operand A and the scales of four sub-blocks at a time, right before their first use (an LDS read is
            // covered by the step in front of it; all eight at once are 16 to 32 registers more, which Q4_K and Q6_K spilled).
            // From the image: everything at the start, in one trip.
            constexpr int kPart = STAGED ? 4 : 8;
            v4i areg[kPart];
            float xs0[kPart], xs1[kPart], xm0[kPart], xm1[kPart];
            auto part_a = [&](int ib0) {
                if constexpr (!EARLY)
#pragma unroll
                for (int i = 0; i < kPart; ++i) areg[i] = *reinterpret_cast<const v4i *>(a_lane + (sb * 8 + ib0 + i) * kStrideA);
            };
            auto part_x = [&](int ib0) {
                auto get = [&](const float * p, float (&v)[kPart]) {
#pragma unroll
                    for (int i = 0; i < kPart; i += 4) {
                        const float4 f = *reinterpret_cast<const float4 *>(p + sb * 8 + ib0 + i);
                        v[i] = f.x; v[i + 1] = f.y; v[i + 2] = f.z; v[i + 3] = f.w;
                    }
                };
                if constexpr (!UNI) { get(sc0, xs0); get(sc1, xs1); }       // activation scales of the sub-blocks
                if constexpr (F::kMin && EARLY) {
                    const float4 f = m_row[0], h = m_row[1];
                    xm0[0] = f.x; xm0[1] = f.y; xm0[2] = f.z; xm0[3] = f.w; xm0[4] = h.x; xm0[5] = h.y; xm0[6] = h.z; xm0[7] = h.w;
                } else if constexpr (F::kMin) { get(sum0, xm0); get(sum1, xm1); }  // and their sums
            };
            // The products of step (sub-block, bank, scale group) + 1 are issued before the sums of this step are read: the
            // matrix pipe's latency passes under the next step's lookups instead of in front of this step's multiply-adds.
            const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            constexpr int G = F::kGroups, kSteps = 8 * NB * G;
            v4i w;
            [[maybe_unused]] v4i found;
            auto operand = [&](int i) {
                if constexpr (EARLY) return a_row[i];
                else return areg[i];
            };
            auto issue = [&](int step) {
                const int ib = step / (NB * G), nb = step / G % NB, grp = step % G;
                if (step % (kPart * NB * G) == 0) part_a(ib);
                if constexpr (FMT == TQMOE_IQ3_S) {   // the next step's look-ups are under way while this step's signs are put on and the sums before are added
                                                      // (64 tokens, top-8 of 256: 164 -> 161.6 us a layer)
                    if (step == 0) found = F::lookup(cur.code[0], cur.rec[0], 0, g, lat);
                    w = F::signed_of(found, cur.code[nb], ib, g);
                    if (step + 1 < kSteps) found = F::lookup(cur.code[(step + 1) % NB], cur.rec[(step + 1) % NB], (step + 1) / NB, g, lat);
                } else if (grp == 0) w = F::decode(cur.code[nb], cur.rec[nb], ib, g, lat);
                if constexpr (G == 1) return __builtin_amdgcn_mfma_i32_32x32x32_i8(operand(ib % kPart), w, zero, 0, 0, 0);
                else {   // operand dwords 0 and 2 are the sub-block's first sixteen weights, 1 and 3 the others
                    const v4i rows4 = operand(ib % kPart);
                    const long a2 = long(uint64_t(uint32_t(rows4[grp])) | uint64_t(uint32_t(rows4[grp + 2])) << 32);
                    const long w2 = long(uint64_t(uint32_t(w[grp])) | uint64_t(uint32_t(w[grp + 2])) << 32);
                    return __builtin_amdgcn_mfma_i32_32x32x16_i8(a2, w2, zero, 0, 0, 0);
                }
            };
            constexpr bool kAhead = UNI;   // the other kernels lose more to the registers of a second result than they gain
            v16i acc = issue(0);
            int si[NB][4];   // (hi, lo) plane sums of the two input rows, weighted by the sub-block scales
            float sm[NB][2];
#pragma unroll
            for (int step = 0; step < kSteps; ++step) {
                const int ib = step / (NB * G), nb = step / G % NB, grp = step % G, ip = ib % kPart;
                if (step % (kPart * NB * G) == 0) part_x(ib);
                v16i ahead = zero;
                if constexpr (kAhead) {
                    if (step + 1 < kSteps) ahead = issue(step + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const typename F::Rec & rec = cur.rec[nb];
                if constexpr (F::kFloat) {
                    const float sc = F::scale(rec, ib, grp);
                    accf[nb][0] = fmaf(float((acc[0] << 7) + acc[1]), UNI ? sc : sc * xs0[ip], accf[nb][0]);
                    if constexpr (kIn == 2) accf[nb][1] = fmaf(float((acc[2] << 7) + acc[3]), UNI ? sc : sc * xs1[ip], accf[nb][1]);
                } else if constexpr (UNI) {
                    // |acc| <= 32 * 128 * 128 = 2^19 and |scale| <= 2^7: 24-bit products, and with a scale per sixteen weights
                    // half the |acc|: sixteen of them stay below 2^30
                    const int ls = F::scale(rec, ib, grp);
#pragma unroll
                    for (int q = 0; q < 2 * kIn; ++q) {
                        si[nb][q] = (ib || grp ? si[nb][q] : 0) + __mul24(acc[q], ls);
                        asm("" : "+v"(si[nb][q]));   // (one multiply-add each: two steps' products are otherwise made apart and added in a third instruction)
                    }
                    if (ib == 7 && grp == G - 1) {
                        const float d = F::d(rec);
                        accf[nb][0] += (float(si[nb][0]) * 128.f + float(si[nb][1])) * d;
                        if constexpr (kIn == 2) accf[nb][1] += (float(si[nb][2]) * 128.f + float(si[nb][3])) * d;
                    }
                } else {
                    const float ws = F::d(rec) * float(F::scale(rec, ib, grp));
                    accf[nb][0] += float((acc[0] << 7) + acc[1]) * (ws * xs0[ip]);
                    accf[nb][1] += float((acc[2] << 7) + acc[3]) * (ws * xs1[ip]);
                }
                if constexpr (F::kMin) {
                    const float mn = F::minimum(rec, ib);
                    sm[nb][0] = ib ? fmaf(mn, xm0[ip], sm[nb][0]) : mn * xm0[ip];
                    if constexpr (kIn == 2) sm[nb][1] = ib ? fmaf(mn, xm1[ip], sm[nb][1]) : mn * xm1[ip];
                    if (ib == 7) {
                        const float dm = F::dmin(rec);
                        accm[nb][0] = fmaf(dm, sm[nb][0], accm[nb][0]);
                        if constexpr (kIn == 2) accm[nb][1] = fmaf(dm, sm[nb][1], accm[nb][1]);
                    }
                }
                // only four of the sixteen result registers are read; the others count as in use until here, or they are handed
                // to the next lookups while the matrix pipe still writes them and every such write waits for the pipe
                asm volatile("" : : "v"(acc));
                if constexpr (kAhead) acc = ahead;
                else if (step + 1 < kSteps) acc = issue(step + 1);
            }
        };
        if constexpr (MULTI) {
            // Several row tiles a wave, one after the other (the launcher has made sure that every wave of the block has the
            // same steps: no ragged tiles, no shorter shared expert): the block finds its input rows and stages them once, and
            // the weight loads run on across the tiles' ends, the next tile's first under this tile's sums.
            const int nsteps = sb_end / wk, total = tl_count * nsteps;
            auto fetch_step = [&](int gs, Cold & c) { fetch_tile(gs / nsteps * tpw, wk_i + gs % nsteps * wk, c); };
            auto after = [&](int gs) {   // step gs is done: was it its tile's last?
                if ((gs + 1) % nsteps) return;
                finish((bx * tl_count + gs / nsteps) * tpw, true);
                clear();
            };
            for (int gs = 0; gs < total; gs += 2) {
                fetch_step(min(gs + 1, total - 1), c1);
                multiply(wk_i + gs % nsteps * wk, c0);
                after(gs);
                if (gs + 1 >= total) break;
                fetch_step(min(gs + 2, total - 1), c0);
                multiply(wk_i + (gs + 1) % nsteps * wk, c1);
                after(gs + 1);
            }
        } else if constexpr (STAGED) {
            const int last = wk_i + (sb_end - 1 - wk_i) / wk * wk;   // the wave's last super-block
            for (int sb = wk_i; sb <= last; sb += 2 * wk) {
                fetch(min(sb + wk, last), c1);
                multiply(sb, c0);
                if (sb + wk > last) break;
                fetch(min(sb + 2 * wk, last), c0);
                multiply(sb + wk, c1);
            }
        } else {   // short batches: most waves have one super-block, and nothing is fetched that is not multiplied
            for (int sb = wk_i; sb < sb_end; sb += wk) {
                if (sb + wk < sb_end) fetch(sb + wk, c1);
                multiply(sb, c0);
                c0 = c1;
                if constexpr (EARLY) if (sb + wk < sb_end) fetch_row(sb + wk);
            }
        }
    }

    if constexpr (!MULTI) finish(bx * tpw, valid);
}

template <uint32_t FMT>
void mfma_launch(int nb, BankView b0, BankView b1, const uint8_t * image, void * out0, void * out1, uint32_t ytype, const int * ids, int A, int xdiv, int mode,
            int slots, int topk, int shared_lim, int gateup, bool uniform, Glu glu, hipStream_t s, DecodeTopk route = DecodeTopk{}) {
    const int NSB = b0.cols / 256, tiles = b0.rows / 32;
    // Waves that share a row's super-blocks: as many as it takes to put a few thousand waves in flight (a short batch
    // is bound by the latency of one wave's chain), fewer when the batch has the waves anyway (a longer chain per
    // wave streams with its loads one super-block ahead and saves the cross-wave sums), and fewer at once where registers
    // leave a SIMD two waves. Shares may differ by a super-block: a row of 11 at one token takes 21 us a layer with four or
    // eight waves and 33 with one (Q4_K, ff 512); with many units an uneven split only loses (nine super-blocks, 5120
    // units: 111 us against 107). Blocks of five to seven waves fill a compute unit badly: only the smallest launches take more
    // than four waves (12 super-blocks, ff 1536: one token, four waves 32 us, six 38; four tokens, two 80, four 79, six 95).
    // One bank, eight tokens of 8 of 128 experts, ff 512 to 1536: one wave a row 55 to 92 us a layer, two 59 to 103.
    const int64_t units = int64_t(A) * tiles;
    const int halves = kDecodeWaves<FMT, 2, true, 0> == 2 && NSB <= 12 ? 576 : 768;   // units of two banks from which two waves share a row
    int wk = nb == 2 ? (units >= 8192 ? 1 : units >= 2048 ? (NSB >= 8 && (NSB % 2 == 0 || units < 3072) ? 2 : 1) : units > halves ? 2 : units >= 320 ? 4 : kMaxWaves)
                     : (units >= 2048 ? 1 : units >= 1024 ? 2 : units >= 320 ? 4 : kMaxWaves);
    if (wk > NSB) wk = NSB;
    const int waves = wk > 4 ? wk : 4;                    // per block: small blocks, a compute unit holds several and their phases interleave
    int tpw = waves / wk;                                                 // row tiles per block
    if (tpw > tiles) tpw = tiles;
    const unsigned threads = unsigned(wk * tpw * 64);
    // dynamic LDS: the partial sums; behind them the input rows' planes (256 bytes per sub-block) and, for rows with a scale per
    // sub-block, the scales
    size_t lds = size_t(wk * tpw) * nb * kTP * 32 * sizeof(float);
    // the input rows go through LDS from a dozen assignments on (the waves then overlap each other's waits, and what
    // counts is that a wave's own weight loads stay in flight under its products: 10 tokens of 8 of 128 experts, Q4_K 71.5
    // and 61.3 us a layer, NVFP4G 69.2 and 68.0, IQ3_S 67.7 and 64.7); a shorter batch is one chain of dependent steps per wave,
    // and the extra stop at a barrier costs more than the exact waits return
    const bool staged = A >= kStagedFrom && !route.logits;
    // ... and a wave then takes up to four row tiles one after the other, as long as the grid keeps five blocks per compute
    // unit: the block's search for its input rows and their staging are paid once for all of them, but a grid of two or
    // three blocks per unit, some of which find their expert taken by another and leave, ends in a round that most units
    // sit out. A Q4_K/Q6_K layer of 23 tokens over 125 experts takes 99 us with two blocks as the least, 90 with five; IQ3_S with
    // 20 tokens over 64 experts 94 and 78. (Not where a shared expert has fewer columns than the others: the waves' steps then
    // differ. 64 tokens, top-8 of 256, without a shared expert: 170 us a layer with one row tile a wave, 164 with four.)
    constexpr int kLeastBlocks = 1280;
    int tl = 1;
    if (staged && nb == 1 && NSB % wk == 0 && (slots <= topk || shared_lim == (gateup ? b0.rows : b0.cols)))
        while (tl < 4 && tiles % (tpw * tl * 2) == 0 && int64_t(tiles / (tpw * tl * 2)) * A >= kLeastBlocks) tl *= 2;
    const unsigned groups = unsigned((tiles + tpw * tl - 1) / (tpw * tl));
    if (route.logits) {
        const int64_t work = int64_t(groups) * A;
        route.groups = int(groups);
        route.per_group = 0xFFFFFFFFu / groups + 1;
        route.apart = (work + 255) / 256 == (work + A / slots + 255) / 256;
    }
    const dim3 grid = route.logits ? dim3(groups * unsigned(slots) + unsigned(route.apart), unsigned(A / slots)) : dim3(groups, unsigned(A));
    const int a_off = int(lds);
    if (staged) lds += size_t(b0.cols / 32) * (256 + ((uniform ? 0 : 1) + (MfmaFormat<FMT>::kMin ? 1 : 0)) * kTP * sizeof(float));
    auto go = [&](auto kernel) { kernel<<<grid, threads, lds, s>>>(b0, b1, image, out0, out1, ytype, ids, A, xdiv, mode, slots, topk, shared_lim, wk, tpw, gateup, a_off, tl, glu, route); };
    if (route.logits) {   // few tokens
        if (route.experts <= 128) go(decode_mfma_k<FMT, 2, true, 0, 2>); else go(decode_mfma_k<FMT, 2, true, 0, 8>);
        return;
    }
    if (nb == 2 && uniform) staged ? go(decode_mfma_k<FMT, 2, true, 1>) : go(decode_mfma_k<FMT, 2, true, 0>);
    else if (nb == 2) staged ? go(decode_mfma_k<FMT, 2, false, 1>) : go(decode_mfma_k<FMT, 2, false, 0>);
    else if (tl > 1) go(decode_mfma_k<FMT, 1, false, 2>);
    else staged ? go(decode_mfma_k<FMT, 1, false, 1>) : go(decode_mfma_k<FMT, 1, false, 0>);
}

// The down product of one to a few tokens and the weighted sum over their experts. A block takes one token and 32 output columns
// (a tile of 32 weight rows in every expert of the token); its waves take (slot, super-block) units in turn, leave each unit's
// 32 sums in LDS, and the block adds a slot's super-blocks, then the slots in order. Against a product launch per assignment
// and a launch that sums: one launch, one trip through memory and the [slots][hidden] fp32 rows less. Few blocks (hidden / 32
// a token), each with all its loads in flight: a chain of one trip to memory and a few hundred instructions.
//
// What bounds it is the vector work of a compute unit (a unit's decode serves one input row, and the blocks are few), so while
// they still find compute units of their own, blocks take half a tile (HALF): the matrix instruction's columns are then sixteen weight rows
// of two sub-blocks, its rows the planes of both sub-blocks' activations, and a lane decodes half as much.
// (2048 columns out, us, whole / half tiles: one token of the 512-expert IQ4_XS layer 7.2 / 5.9, of Q4_K top-8 6.9 / 5.8, of NVFP4G 7.4 /
// 6.1; two tokens, 256 half tiles, 7.0 / 5.8; three tokens, 384 half tiles on 256 compute units, 7.7 / 10.5.)
constexpr int kHalfBlocks = 256, kDownWaves = 16;
template <uint32_t FMT, bool HALF>
__global__ __launch_bounds__(64 * kDownWaves) void down_combine_k(DownCombineArgs k) {
    using F = MfmaFormat<FMT>;
    constexpr int kRows = HALF ? 16 : 32, kSub = HALF ? 4 : 8, kStep = HALF ? 2 : 1;   // weight rows of a block; products of a unit; sub-blocks of one
    extern __shared__ float part[];   // [units][32] sums, then [slots][kRows] weighted rows
    __shared__ uint32_t lat[F::kLattice];
    const int token = blockIdx.y, tile = blockIdx.x / (32 / kRows), S = k.b.cols / 32, NSB = S / 8, tiles = k.b.rows / 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 31, g = lane >> 5;
    const int odd = HALF ? n >> 4 : 0, row_n = HALF ? int(blockIdx.x & 1) * 16 + (n & 15) : n;   // the lane's sub-blocks, its weight row in the tile
    const int shared_sb = k.slots > k.topk ? k.shared_cols / 256 : 0, units = k.topk * NSB + shared_sb;
    const int extra = k.experts - 1;                           // the shared expert's place
    struct Unit { typename F::Codes code; typename F::Rec rec; v4i a[kSub]; float4 xs[2], xm[2]; float rf; };
    auto slot_of = [&](int u) { return min(NSB == 1 ? u : int(__umulhi(uint32_t(u), k.per_slot)), k.slots - 1); };
    auto fetch = [&](int u, int slot, int e, Unit & c) {
        const int sb = u - slot * NSB;
        const uint8_t * row = image_row_ptr(k.image, int64_t(token) * k.slots + slot, S);
        const uint8_t * a = row + sb * 512 + (HALF ? ((n >> 1) & 1) * 64 : 0) + (n & 1) * 32 + g * 16;
#pragma unroll
        for (int i = 0; i < kSub; ++i) c.a[i] = *reinterpret_cast<const v4i *>(a + i * kStep * 64);
        const float4 * xs = reinterpret_cast<const float4 *>(image_scales(row, S) + sb * 8);
        c.xs[0] = xs[0]; c.xs[1] = xs[1];
        if constexpr (F::kMin) { const float4 * xm = reinterpret_cast<const float4 *>(image_sums(row, S) + sb * 8); c.xm[0] = xm[0]; c.xm[1] = xm[1]; }
        e = min(max(e, 0), extra);   // an id outside the bank: a bank's weights, not added below
        const int64_t at = (int64_t(e) * tiles + tile) * NSB + sb;
        if constexpr (HALF) F::half_codes(k.b.codes + at * F::kCodeBytes, row_n, g, odd, c.code);
        else F::codes(k.b.codes + at * F::kCodeBytes, n, g, c.code);
        c.rec = F::rec(k.b.aux + at * F::kRecBytes, row_n);
        c.rf = F::row_factor(k.b, (int64_t(e) * k.b.rows) + tile * 32 + row_n);
    };
    auto multiply = [&](const Unit & c) {
        const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        auto of_lane = [&](const float4 (&v)[2], int i) {      // sub-block kStep i + odd
            const float w[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
            return HALF ? (odd ? w[kStep * i + kStep - 1] : w[kStep * i]) : w[i];
        };
        typename F::Rec rec = c.rec;
        if constexpr (HALF) rec = F::odd_rec(c.rec, odd);
        float sum = 0.f, mins = 0.f;
#pragma unroll
        for (int i = 0; i < kSub; ++i) {
            const int ib = kStep * i;
            const float xs = of_lane(c.xs, i);
            const v4i w = F::decode(c.code, rec, ib, g, lat);
            // (every even row of operand A is the hi plane of the one input row, every odd one the lo plane; HALF: rows 0 and 1 those
            // of the even sub-block, 2 and 3 those of the odd one)
            auto add = [&](const v16i & acc, int grp) {
                const int hi = odd ? acc[2] : acc[0], lo = odd ? acc[3] : acc[1];
                sum += float((hi << 7) + lo) * (F::d(c.rec) * float(F::scale(rec, ib, grp)) * xs);
                asm volatile("" : : "v"(acc));   // (all sixteen registers in use until here: see decode_mfma_k)
            };
            if constexpr (F::kGroups == 1) add(__builtin_amdgcn_mfma_i32_32x32x32_i8(c.a[i], w, zero, 0, 0, 0), 0);
            else
#pragma unroll
                for (int grp = 0; grp < 2; ++grp) {
                    const long a2 = long(uint64_t(uint32_t(c.a[i][grp])) | uint64_t(uint32_t(c.a[i][grp + 2])) << 32);
                    const long w2 = long(uint64_t(uint32_t(w[grp])) | uint64_t(uint32_t(w[grp + 2])) << 32);
                    add(__builtin_amdgcn_mfma_i32_32x32x16_i8(a2, w2, zero, 0, 0, 0), grp);
                }
            if constexpr (F::kGroups == 2) __builtin_amdgcn_sched_barrier(0);   // (sixteen results under way are more than the registers hold)
            if constexpr (F::kMin) mins = fmaf(F::minimum(rec, ib), of_lane(c.xm, i), mins);
        }
        if constexpr (F::kMin) sum = fmaf(-F::dmin(c.rec), mins, sum);
        return sum * c.rf;
    };
    if constexpr (FMT == TQMOE_IQ3_S) {
        F::lattice(lat, threadIdx.x, blockDim.x);
        __syncthreads();
    }
    // (a second unit's loads in flight under the first's products: the registers of a block of sixteen waves spill, 7.9 -> 23.7 us
    // for Q4_K at one token)
    // what the sums need at the end, on its way meanwhile (Q6_K's whole tiles have no registers for it)
    const int sums = k.slots * kRows;
    auto weight_of = [&](int slot) { return slot < k.topk ? k.weights[token * k.topk + slot] : k.shared_weights[token]; };
    const int64_t o = int64_t(token) * k.b.rows + int64_t(blockIdx.x) * kRows + threadIdx.x;
    [[maybe_unused]] float first_w = 0.f;
    [[maybe_unused]] uint16_t res = 0;
    if constexpr (HALF) {
        if (int(threadIdx.x) < sums) first_w = weight_of(threadIdx.x / kRows);
        if (k.residual && k.otype != TQMOE_F32 && threadIdx.x < kRows) res = k.residual[o];
    }
    for (int u = wave; u < units; u += kDownWaves) {
        const int slot = slot_of(u), e = slot < k.topk ? k.ids[token * k.topk + slot] : extra;
        Unit c;
        fetch(u, slot, e, c);
        if constexpr (!HALF && F::kGroups == 2) __builtin_amdgcn_sched_barrier(0);   // (or the decode is moved up between the loads, and Q6_K spills: one token 32 -> 82 us a layer)
        const float v = multiply(c);
        if (g == 0) part[u * 32 + n] = e >= 0 && e <= extra ? v : 0.f;
    }
    __syncthreads();
    float * rows = part + units * 32;
    for (int i = threadIdx.x; i < sums; i += blockDim.x) {
        const int slot = i / kRows, nsb = slot < k.topk ? NSB : shared_sb;
        float v = 0.f;
        for (int sb = 0; sb < nsb; ++sb)
            for (int h = 0; h < 32 / kRows; ++h) v += part[(slot * NSB + sb) * 32 + h * kRows + i % kRows];
        rows[i] = (HALF && i == int(threadIdx.x) ? first_w : weight_of(slot)) * v;
    }
    __syncthreads();
    if (threadIdx.x < kRows) {
        float sum = 0.f;
        for (int s = 0; s < k.slots; ++s) sum += rows[s * kRows + threadIdx.x];
        if (k.otype == TQMOE_F32) static_cast<float *>(k.out)[o] = sum;
        else {
            if (k.residual) sum = bf16_bits_to_float(float_to_bf16_bits(sum)) + bf16_bits_to_float(HALF ? res : k.residual[o]);
            static_cast<uint16_t *>(k.out)[o] = float_to_bf16_bits(sum);
        }
    }
}

template <uint32_t FMT> void down_combine_launch(DownCombineArgs k, hipStream_t s) {
    const int NSB = k.b.cols / 256;
    k.experts = int(k.b.rows_total / k.b.rows);
    k.per_slot = 0xFFFFFFFFu / uint32_t(NSB) + 1;
    const int units = k.topk * NSB + (k.slots > k.topk ? k.shared_cols / 256 : 0);
    const size_t lds = size_t(units + k.slots) * 32 * sizeof(float);
    if (int64_t(k.n) * (k.b.rows / 16) <= kHalfBlocks) down_combine_k<FMT, true><<<dim3(unsigned(k.b.rows / 16), unsigned(k.n)), 64 * kDownWaves, lds, s>>>(k);
    else down_combine_k<FMT, false><<<dim3(unsigned(k.b.rows / 32), unsigned(k.n)), 64 * kDownWaves, lds, s>>>(k);
}

// the shapes the kernel takes: whole tiles, whole super-blocks (a narrower shared expert included)
inline bool mfma_takes(int rows, int cols, int shared_cols) { return rows % 32 == 0 && cols % 256 == 0 && shared_cols % 256 == 0; }

}  // namespace
}  // namespace tqmoe
