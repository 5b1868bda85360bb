// Grouped fp16 products of the tile-major bank formats (IQ4_XS, Q4_K, Q6_K, IQ3_S) at prefill sizes, on prepared rows.
//
// A block of four waves takes one item of the plan (an expert and up to 128 of its input rows) and eight tiles of 32 weight
// rows, two a wave: the same tile of the gate and the up bank, or two tiles of one bank. Per stage of 64 weights of a row:
//  * input rows (fp16, in the order the weight operands come in: operand_pos) and the weights' code bytes go straight from
//    memory to LDS one stage ahead of their use (16 bytes a lane, no registers, no vector instructions); one barrier a
//    stage;
//  * lane (n, g) of a wave turns the codes of sub-block g of weight row n into the sixteen dwords of halves that are
//    operand B of the stage's four matrix instructions per row tile: weights never exist as halves in LDS;
//  * the matrix instructions of code dword j are followed by the decode of dword j of the next stage into the same
//    registers, six or so vector instructions to a matrix instruction.
//
// Weight values. A code's table value (or the code itself) lands in the low byte of the half 1024 + u by one byte permute
// or mask per pair; one mixed-precision multiply-add per weight takes the bias off and puts the fp32 scale (and minimum)
// on, one conversion per pair rounds to fp16: 19 (Q4_K) to 27 (IQ4_XS) vector instructions for eight weights, one rounding.
// (Packed fp16 multiply-adds take four fewer and round twice: a quarter more error in the layer's result.)
//
// Rows per item: a weight is decoded once per item and wave, so 128 rows spread its 23 / 8 instructions a weight over four
// matrix instructions; with the two banks' eight accumulators (128 registers) two waves fit a SIMD, and one of them decodes
// while the other's products run. Items of one and two row tiles have loops of their own with fewer products.
#pragma once
#include "decode_api.cuh"
#include "decode_table.cuh"
#include "formats.cuh"
#include "grouped_f16_api.cuh"

namespace tqmoe {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

// 16 bytes a lane from memory to LDS at `lds` (a wave-uniform byte address) + 16 * lane. The compiler does not count these:
// dma_wait() before the barrier that publishes them.
__device__ __forceinline__ void dma16(const void * p, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(p), "s"(lds) : "memory");
}
__device__ __forceinline__ void dma_wait_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ uint32_t lds_address(const void * p) {
    return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint8_t *)(p)));
}

__device__ __forceinline__ v2h as_h2(uint32_t v) { return __builtin_bit_cast(v2h, v); }
__device__ __forceinline__ uint32_t bits_of(v2h v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ v2h both(float v) { const _Float16 h = _Float16(v); return v2h{h, h}; }
__device__ __forceinline__ v2h both_bits(uint32_t h16) { return as_h2(h16 | h16 << 16); }
// both halves of u times s plus c, in fp32, rounded to halves: two v_fma_mix_f32 and a packed conversion (v_fma_mixlo_f16 and
// v_fma_mixhi_f16 do it in two, at half the rate)
__device__ __forceinline__ uint32_t mix2(v2h u, float s, float c) {
    const float lo = fmaf(float(u[0]), s, c), hi = fmaf(float(u[1]), s, c);
    return bits_of(v2h{_Float16(lo), _Float16(hi)});
}
// bytes 0, 2 and bytes 1, 3 of u as halves 1024 + byte
__device__ __forceinline__ v2h bias_even(uint32_t u) { return as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04020400u)); }
__device__ __forceinline__ v2h bias_odd(uint32_t u) { return as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030401u)); }

// What the kernel needs of a format.
// kCodes: 1 KB transfers a bank and stage (64 lanes x 16 bytes), their lane's source at stage 0 in code(), kCodeStep
// bytes from stage to stage inside a super-block and kCodeJump more at its end. kRecs transfers for both banks' records
// of the stage's super-block: rec(). Prep: what decoding a stage needs in registers; slice(): operand B of code dword j.
template <uint32_t FMT> struct GroupedFormat;

struct GroupedNibbles {   // 16 code bytes a sub-block in the canonical order
    static constexpr int kCodes = 1, kRecs = 1;
    static __device__ __forceinline__ const uint8_t * code(const BankView & b, int64_t tile, int S, int, int lane) { return b.codes + tile * S * 512 + lane * 16; }
    static __device__ __forceinline__ int code_at(int, int st) { return st * 1024; }
};

template <> struct GroupedFormat<TQMOE_IQ4_XS> : GroupedNibbles {
    static constexpr int kLattice = 1;
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int, int lane) {
        const int l = lane & 31;   // sixteen lanes a bank; the upper half of the wave repeats the lower
        return (l < 16 ? b0.aux + tile0 * (S / 8) * 256 : b1.aux + tile1 * (S / 8) * 256) + (l & 15) * 16;
    }
    static constexpr int kRecStep = 256;
    struct Prep { uint32_t c[4]; float s, off; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint2 *, Prep & p) {
        const uint4 c = *reinterpret_cast<const uint4 *>(w + nb * 1024 + g * 512 + n * 16);
        const uint2 r = *reinterpret_cast<const uint2 *>(w + 2048 + nb * 256 + n * 8);
        p.c[0] = c.x; p.c[1] = c.y; p.c[2] = c.z; p.c[3] = c.w;
        p.s = half_bits_to_float(iq4xs_d_bits(r)) * float(iq4xs_lsm32(r, (2 * st + g) & 7));   // 17 bits: exact
        p.off = p.s * -1152.f;                                                                 // four more: exact
    }
    static __device__ __forceinline__ uint4 slice(const Prep & p, int j) {
        constexpr Table16 t = table16({1, 24, 45, 63, 79, 93, 106, 118, 129, 141, 153, 166, 181, 197, 217, 241});   // the values + 128
        const uint32_t c = p.c[j], lo = pick(t, c & 0x0F0F0F0Fu), hi = pick(t, (c >> 4) & 0x0F0F0F0Fu);
        return make_uint4(mix2(bias_even(lo), p.s, p.off), mix2(bias_odd(lo), p.s, p.off), mix2(bias_even(hi), p.s, p.off), mix2(bias_odd(hi), p.s, p.off));
    }
};

template <> struct GroupedFormat<TQMOE_Q4_K> : GroupedNibbles {
    static constexpr int kLattice = 1;
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int, int lane) {
        return (lane < 32 ? b0.aux + tile0 * (S / 8) * 512 : b1.aux + tile1 * (S / 8) * 512) + (lane & 31) * 16;
    }
    static constexpr int kRecStep = 512;
    struct Prep { uint32_t c[4]; float s, off; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint2 *, Prep & p) {
        const uint4 c = *reinterpret_cast<const uint4 *>(w + nb * 1024 + g * 512 + n * 16);
        const uint4 r = *reinterpret_cast<const uint4 *>(w + 2048 + nb * 512 + n * 16);
        p.c[0] = c.x; p.c[1] = c.y; p.c[2] = c.z; p.c[3] = c.w;
        int sc, mn;
        q4k_scale_min_flat(r.y, r.z, r.w, (2 * st + g) & 7, sc, mn);
        p.s = half_bits_to_float(uint16_t(r.x & 0xFFFFu)) * float(sc);
        // the bias and the minimum in one constant: its rounding is 2^-15 of a code step
        p.off = -fmaf(p.s, 1024.f, half_bits_to_float(uint16_t(r.x >> 16)) * float(mn));
    }
    static __device__ __forceinline__ uint4 slice(const Prep & p, int j) {
        const uint32_t c = p.c[j];
        uint32_t mask = 0x000F000Fu;
        asm("" : "+v"(mask));                      // in a register, so that mask and bias are one instruction
        auto val = [&](uint32_t x) { return mix2(as_h2((x & mask) | 0x64006400u), p.s, p.off); };
        return make_uint4(val(c), val(c >> 8), val(c >> 4), val(c >> 12));
    }
};

template <> struct GroupedFormat<TQMOE_Q6_K> {
    static constexpr int kCodes = 2, kRecs = 2, kLattice = 1;
    static __device__ __forceinline__ const uint8_t * code(const BankView & b, int64_t tile, int S, int i, int lane) {   // low nibbles; upper bits of the pair (twice)
        const uint8_t * q = b.codes + tile * (S / 8) * 6144;
        return i == 0 ? q + lane * 16 : q + 4096 + (lane & 31) * 16;
    }
    static __device__ __forceinline__ int code_at(int i, int st) { return (st >> 2) * 6144 + (st & 3) * (i == 0 ? 1024 : 512); }
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int i, int lane) {
        return (i == 0 ? b0.aux + tile0 * (S / 8) * 1024 : b1.aux + tile1 * (S / 8) * 1024) + lane * 16;
    }
    static constexpr int kRecStep = 1024;
    struct Prep { uint32_t lo[4], hi[2]; float s[2], off[2]; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint2 *, Prep & p) {
        const uint4 c = *reinterpret_cast<const uint4 *>(w + nb * 2048 + g * 512 + n * 16);
        p.lo[0] = c.x; p.lo[1] = c.y; p.lo[2] = c.z; p.lo[3] = c.w;
        p.hi[0] = *reinterpret_cast<const uint32_t *>(w + nb * 2048 + 1024 + n * 16 + g * 4);
        p.hi[1] = *reinterpret_cast<const uint32_t *>(w + nb * 2048 + 1024 + n * 16 + 8 + g * 4);
        const uint8_t * r = w + 4096 + nb * 1024 + n * 32;
        const uint32_t s2 = *reinterpret_cast<const uint16_t *>(r + 2 * ((2 * st + g) & 7));
        const float d = 0.25f * half_bits_to_float(*reinterpret_cast<const uint16_t *>(r + 16));   // the operand byte is four times the value
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            p.s[i] = d * float(int(__builtin_amdgcn_sbfe(int(s2), 8 * i, 8)));
            p.off[i] = p.s[i] * -1152.f;           // 18 bits and four: exact
        }
    }
    static __device__ __forceinline__ uint4 slice(const Prep & p, int j) {
        // dword j of the low nibbles: half j / 2 of the sub-block, its operand dwords 2 (j % 2) and + 1
        const uint32_t lo = p.lo[j], hi = p.hi[j >> 1] >> (4 * (j & 1));
        const uint32_t a = ((lo << 2) & 0x3C3C3C3Cu) | ((hi << 6) & 0xC0C0C0C0u), b = ((lo >> 2) & 0x3C3C3C3Cu) | ((hi << 4) & 0xC0C0C0C0u);
        auto val = [&](v2h u, int i) { return mix2(u, p.s[i], p.off[i]); };
        const uint32_t ua = a ^ 0x80808080u, ub = b ^ 0x80808080u;
        return make_uint4(val(bias_even(ua), 0), val(bias_odd(ua), 0), val(bias_even(ub), 1), val(bias_odd(ub), 1));
    }
};

template <> struct GroupedFormat<TQMOE_IQ3_S> {
    static constexpr int kCodes = 1, kRecs = 1, kLattice = 512;
    static __device__ __forceinline__ const uint8_t * code(const BankView & b, int64_t tile, int S, int, int lane) {   // the pair's indices, then the signs
        return b.codes + tile * (S / 8) * 3072 + (lane < 32 ? 0 : 2048) + (lane & 31) * 16;
    }
    // (indices: 512 bytes a pair, signs: 512 bytes two pairs; the lane's own step)
    static __device__ __forceinline__ int code_at(int, int st) { return (st >> 2) * 3072 + ((threadIdx.x & 32) ? ((st & 3) >> 1) * 512 : (st & 3) * 512); }
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int, int lane) {
        return (lane < 32 ? b0.aux + tile0 * (S / 8) * 512 : b1.aux + tile1 * (S / 8) * 512) + (lane & 31) * 16;
    }
    static constexpr int kRecStep = 512;
    struct Prep { uint32_t qs[2], sg, qh; v2h sc, d; const uint2 * lat; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint2 * lat, Prep & p) {
        const uint8_t * q = w + nb * 1024 + n * 16;
        p.qs[0] = *reinterpret_cast<const uint32_t *>(q + g * 4);
        p.qs[1] = *reinterpret_cast<const uint32_t *>(q + 8 + g * 4);
        const int ib = (2 * st + g) & 7;
        p.sg = *reinterpret_cast<const uint32_t *>(q + 512 + (ib & 3) * 4);
        const uint4 r = *reinterpret_cast<const uint4 *>(w + 2048 + nb * 512 + n * 16);
        p.qh = (ib < 4 ? r.y : r.z) >> (8 * (ib & 3));
        const uint32_t ls = (ib < 4 ? r.x >> (16 + 4 * ib) : r.w >> (4 * (ib - 4))) & 15u;
        p.sc = both(float(1 + 2 * int(ls)));
        p.d = both_bits(r.x & 0xFFFFu);
        p.lat = lat;
    }
    static __device__ __forceinline__ uint4 slice(const Prep & p, int j) {
        const int h = j >> 1, q = 2 * (j & 1);     // operand dwords q and q + 1 of half h: weights 4 j .. and 16 + 4 j ..
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t idx = ((p.qs[h] >> (8 * (q + i))) & 0xFFu) | ((p.qh << (8 - 4 * h - q - i)) & 0x100u);
            const uint2 mag = p.lat[idx];          // the four magnitudes as halves, weights 0, 2 and 1, 3
            const int s = 4 * h + q + i;           // bit 8 t + s: the sign of weight t
            // times the integer scale (exact), times d (the one rounding)
            v[2 * i] = bits_of(as_h2(mag.x ^ ((p.sg << (15 - s)) & 0x80008000u)) * p.sc * p.d);
            v[2 * i + 1] = bits_of(as_h2(mag.y ^ ((p.sg << (7 - s)) & 0x80008000u)) * p.sc * p.d);
        }
        return make_uint4(v[0], v[1], v[2], v[3]);
    }
};

// bytes of a wave's codes and records of one stage
template <class W> constexpr int kStageW = 2 * W::kCodes * 1024 + W::kRecs * 1024;
template <class W> constexpr int grouped_f16_lds(int mt) { return 2 * mt * 4096 + 4 * 2 * kStageW<W>; }

template <uint32_t FMT, bool GATEUP, class OT>
__global__ __launch_bounds__(256, 2) void grouped_f16_k(GroupedF16Args k) {
    using W = GroupedFormat<FMT>;
    constexpr int MTMAX = kGroupedRows / 32;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];   // [2][MTMAX * 4096] input rows | [4 waves][2][kStageW] codes and records
    __shared__ uint2 s_lat[W::kLattice];
    __shared__ int s_asg[kGroupedRows];
    __shared__ float s_scale[kGroupedRows];
    // Items that share input rows (an item of the plan, all its groups of weight tiles) run on one XCD, one after the other.
    const int xcd = int(blockIdx.x) & 7, at = int(blockIdx.x) >> 3;
    const int chunk = at / k.groups * 8 + xcd, grp = at % k.groups;
    if (chunk >= k.plan[0].x) return;
    const int4 item = k.plan[1 + chunk];           // expert, its first row in perm, rows
    const int e = item.x, cnt = item.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 31, g = lane >> 5;
    const int rows = k.b0.rows, cols = k.b0.cols, S = cols / 32, tiles = rows / 32;
    const bool is_shared = e == k.shared_expert;
    const int row_lim = GATEUP && is_shared ? k.shared_lim : rows;
    const int stages = (!GATEUP && is_shared ? k.shared_lim : cols) / 64;
    if constexpr (W::kLattice > 1)
        for (int i = tid; i < W::kLattice; i += 256) {
            const v2h bias = as_h2(0xE400E400u);       // -1024
            const uint32_t m = d_iq3s_grid.v[i];
            s_lat[i] = make_uint2(bits_of(bias_even(m) + bias), bits_of(bias_odd(m) + bias));
        }
    if (tid < kGroupedRows) {
        s_asg[tid] = tid < cnt ? k.perm[item.y + tid] : -1;
        s_scale[tid] = 1.f;
        if (k.xs && tid < cnt) s_scale[tid] = k.xs[s_asg[tid] / k.xdiv];
    }
    __syncthreads();
    // weight tiles of this wave (past the last one: it once more, not stored)
    int wt[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) wt[b] = GATEUP ? grp * 4 + wave : grp * 8 + wave * 2 + b;

    auto body = [&](auto tag) {
        constexpr int MT = decltype(tag)::value;
        v16f acc[2][MT];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[b][m][i] = 0.f;
        const bool any = GATEUP ? grp * 128 < row_lim : true;
        if (any) {
            // input rows: transfer q of a wave is rows 8 (4 q + wave) .. + 7 of the stage's 128 bytes, a row's piece p in slot
            // p ^ (row & 7), so that the operand reads (a row a lane) find eight rows' pieces in eight different bank groups
            const uint8_t * a_src[MT];
#pragma unroll
            for (int q = 0; q < MT; ++q) {
                const int row = (4 * q + wave) * 8 + (lane >> 3);
                a_src[q] = reinterpret_cast<const uint8_t *>(k.x) + (int64_t(max(s_asg[row], 0)) / k.xdiv * cols) * 2 + ((lane & 7) ^ (row & 7)) * 16;
            }
            const uint32_t lds0 = lds_address(lds);
            uint8_t * const w_lds = lds + 2 * MTMAX * 4096 + wave * 2 * kStageW<W>;
            const uint32_t w_lds0 = lds_address(w_lds);
            const int64_t t0 = int64_t(e) * tiles + min(wt[0], tiles - 1), t1 = int64_t(e) * tiles + min(wt[1], tiles - 1);
            const uint8_t * c_src[2][W::kCodes], * r_src[W::kRecs];
#pragma unroll
            for (int i = 0; i < W::kCodes; ++i) { c_src[0][i] = W::code(k.b0, t0, S, i, lane); c_src[1][i] = W::code(k.b1, t1, S, i, lane); }
#pragma unroll
            for (int i = 0; i < W::kRecs; ++i) r_src[i] = W::rec(k.b0, k.b1, t0, t1, S, i, lane);
            auto send_a = [&](int st) {
#pragma unroll
                for (int q = 0; q < MT; ++q) dma16(a_src[q] + st * 128, lds0 + (st & 1) * MTMAX * 4096 + (4 * q + wave) * 1024);
            };
            auto send_w = [&](int st) {
                const uint32_t to = w_lds0 + (st & 1) * kStageW<W>;
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < W::kCodes; ++i) dma16(c_src[b][i] + W::code_at(i, st), to + (b * W::kCodes + i) * 1024);
#pragma unroll
                for (int i = 0; i < W::kRecs; ++i) dma16(r_src[i] + (st >> 2) * W::kRecStep, to + (2 * W::kCodes + i) * 1024);
            };
            const uint8_t * a_row = lds + n * 128;
            uint4 bw[2][4];
            typename W::Prep pr[2];
            send_w(0);
            send_a(0);
            dma_wait_barrier();
            if (stages > 1) send_w(1);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                W::prep(w_lds, b, 0, n, g, s_lat, pr[b]);
#pragma unroll
                for (int j = 0; j < 4; ++j) bw[b][j] = W::slice(pr[b], j);
            }
            for (int st = 0; st < stages; ++st) {
                // this stage's rows and the next one's codes are here, and every wave is done with the buffers that are filled now
                if (st) dma_wait_barrier(); else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                if (st + 1 < stages) send_a(st + 1);
                if (st + 2 < stages) send_w(st + 2);
                const int nx = min(st + 1, stages - 1);   // past the last stage: its codes again, not used
#pragma unroll
                for (int b = 0; b < 2; ++b) W::prep(w_lds + (nx & 1) * kStageW<W>, b, nx, n, g, s_lat, pr[b]);
                const uint8_t * a_buf = a_row + (st & 1) * MTMAX * 4096;
                v8h a[2][MT];
                auto read_a = [&](int j) {
#pragma unroll
                    for (int m = 0; m < MT; ++m) a[j & 1][m] = *reinterpret_cast<const v8h *>(a_buf + m * 4096 + (((4 * g + j) ^ (n & 7)) * 16));
                };
                read_a(0);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j < 3) read_a(j + 1);
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int m = 0; m < MT; ++m) acc[b][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[j & 1][m], __builtin_bit_cast(v8h, bw[b][j]), acc[b][m], 0, 0, 0);
#pragma unroll
                    for (int b = 0; b < 2; ++b) bw[b][j] = W::slice(pr[b], j);
                }
            }
        }
        // result register i of lane half g: input row 8 (i / 4) + 4 g + i % 4 of the row tile, weight row n of the weight tile
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            int asg[16];
            float scl[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) { const int r = m * 32 + 8 * (i >> 2) + 4 * g + (i & 3); asg[i] = s_asg[r]; scl[i] = s_scale[r]; }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (asg[i] < 0) continue;
                OT * o = static_cast<OT *>(k.out) + int64_t(asg[i]) * rows;
                auto put = [&](int col, float v) {
                    if constexpr (sizeof(OT) == 4) o[col] = v;
                    else o[col] = __half_as_ushort(__float2half_rn(v));
                };
                if constexpr (GATEUP) {
                    if (wt[0] >= tiles) continue;
                    float gv = acc[0][m][i] * scl[i], uv = acc[1][m][i] * scl[i];
                    glu_clamp_inputs(k.glu, gv, uv);
                    const float v = glu_clamp_silu(k.glu, gv * __builtin_amdgcn_rcpf(1.f + __expf(-gv))) * uv;
                    put(wt[0] * 32 + operand_pos(n), wt[0] * 32 < row_lim ? v : 0.f);
                } else {
#pragma unroll
                    for (int b = 0; b < 2; ++b) if (wt[b] < tiles) put(wt[b] * 32 + n, acc[b][m][i] * scl[i]);
                }
            }
        }
    };
    if (cnt <= 32) body(std::integral_constant<int, 1>{});
    else if (cnt <= 64) body(std::integral_constant<int, 2>{});
    else body(std::integral_constant<int, MTMAX>{});
}

template <uint32_t FMT> void grouped_f16_launch(const GroupedF16Args & k, bool gateup, bool f32_out, unsigned blocks, hipStream_t s) {
    using W = GroupedFormat<FMT>;
    constexpr int bytes = grouped_f16_lds<W>(kGroupedRows / 32);
    auto go = [&](auto kernel) {
        allow_dynamic_lds(reinterpret_cast<const void *>(kernel), bytes);
        kernel<<<blocks, 256, bytes, s>>>(k);
    };
    if (gateup) go(&grouped_f16_k<FMT, true, uint16_t>);
    else if (f32_out) go(&grouped_f16_k<FMT, false, float>);
    else go(&grouped_f16_k<FMT, false, uint16_t>);
}

}  // namespace
}  // namespace tqmoe
