// Grouped products of the tile-major bank formats at prefill sizes, on prepared rows: fp16 operands (IQ4_XS, Q4_K, Q6_K,
// IQ3_S) or E4M3 operands (NVFP4G).
//
// A block of four waves takes one item of the plan (an expert and up to 128 of its input rows) and eight tiles of 32 weight
// rows, two a wave: the same tile of the gate and the up bank, or two tiles of one bank. Per stage (128 bytes of an input row:
// 64 halves or 128 E4M3 values):
//  * input rows (in the order the weight operands come in) and the weights' code bytes go straight from memory to LDS one
//    stage ahead of their use (16 bytes a lane, no registers, no vector instructions); one barrier a stage;
//  * lane (n, g) of a wave turns the codes of sub-block g (E4M3: sub-blocks g and 2 + g) of weight row n into the sixteen
//    dwords that are operand B of the stage's four (two) matrix instructions per row tile: decoded weights never pass
//    through LDS;
//  * the matrix instructions of operand piece j are followed by the decode of piece j of the next stage into the same
//    registers, six or so vector instructions to a matrix instruction.
//
// Weight values. A code's table value lands in the low byte of the half 1024 + u by one byte permute per pair; one
// mixed-precision multiply-add per weight takes the bias off and puts the fp32 scale (and minimum) on, one conversion per
// pair rounds to fp16: 17 (Q4_K, whose codes are halves where they stand) to 27 (IQ4_XS) vector instructions for eight
// weights, one rounding.
// (Packed fp16 multiply-adds take four fewer and round twice: a quarter more error in the layer's result.)
// NVFP4G: the eight magnitudes of a scale byte, rounded to E4M3, are a table in LDS (2 KB for all scales), the code's sign is
// put on beside the look-up; eight instructions for eight weights.
//
// Rows per item: a weight is decoded once per item and wave, so 128 rows spread its instructions over four matrix
// instructions; with the two banks' eight accumulators (128 registers) two waves fit a SIMD, and one of them decodes while
// the other's products run. Items of one and two row tiles have loops of their own with fewer products.
//
// What bounds it (counters: profiles/grouped_rows_counters.txt, of a card on which these launches take 5 % longer): Q4_K, 4096 tokens of 8 experts of 64, gate / up (206 GFLOP): 228 us, 0.90
// PFLOP/s, matrix pipe 48 % busy, vector pipe 53 % (262 us with biased codes; without the decode 205, without the row reads as
// well 178, where a large fp16 product on this card would take 170); NVFP4G, 8192 tokens, gate / up (2.1 TFLOP with down): 808 us,
// 49 % and 52 % (880, 43 % and 55 % with the sign in the table of a scale's weights). A product holds its SIMD's vector issue for about 18 cycles besides its own time, so that a stage's decode does not
// pass under its products for free.
// Items of one row tile are bound by the decode (IQ3_S, 512 tokens: gate / up 117 us, 2.9 TB/s of codes, vector pipe 65 %, LDS 52 %,
// three fifths of that bank conflicts of the lattice's look-ups).
//
// Items of up to kFold row tiles (IQ4_XS and Q6_K: two, IQ3_S: one): the operands are the codes times the integer scale, and every 256
// columns the fp32 sums are multiplied by the super-block's factor instead (the weights are the second operand there, so that a
// lane's factor is its own weight row's). IQ3_S: exact in fp16, 32 of 224 vector instructions a stage less for 16 more, and a rounding
// fewer (the error against float64 5.2e-4 without, 3.6e-4 so). IQ4_XS and Q6_K: bias and scale are whole numbers that halves hold, so that
// one packed multiply-add, rounded once, does for a pair of weights what two mixed ones and a conversion do: eight instructions fewer
// for eight weights, 64 a stage for the 16 (the error 5.2e-4 / 4.6e-4). The sums of both kinds are rounded differently, by 3 to 5.5e-4 of a
// result's norm, so that the loops of one kernel are all of one kind: a row's bits do not say how many rows its expert has from other
// tokens. The second set of sums leaves two row tiles two waves a SIMD in place of three; four have no registers for it. Layer in us, items of
// 64 rows, whole weights / factor outside: 77 experts with 30 rows on average IQ4_XS 181 / 177 (Zipf 178 / 174), Q6_K 203 / 198 (205 / 199), IQ3_S 179
// / 183 (180 / 185). (Two row tiles with one weight tile after the other keep three waves and read the rows twice: level where most items have
// one row tile, 4 to 15 % slower under Zipf.)
#pragma once
#include <type_traits>

#include "decode_api.cuh"
#include "decode_table.cuh"
#include "formats.cuh"
#include "grouped_rows_api.cuh"
#include "lds_dma.cuh"

namespace tqmoe {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

typedef int v8i __attribute__((ext_vector_type(8)));
__device__ __forceinline__ v8i join(uint4 a, uint4 b) { return v8i{int(a.x), int(a.y), int(a.z), int(a.w), int(b.x), int(b.y), int(b.z), int(b.w)}; }
__device__ __forceinline__ v2h as_h2(uint32_t v) { return __builtin_bit_cast(v2h, v); }
__device__ __forceinline__ uint32_t bits_of(v2h v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ v2h both(float v) { const _Float16 h = _Float16(v); return v2h{h, h}; }
__device__ __forceinline__ v2h both_bits(uint32_t h16) { return as_h2(h16 | h16 << 16); }
// both halves of u times s plus c, in fp32, rounded to halves: two v_fma_mix_f32 and a packed conversion, 6.1 ns a SIMD
// (v_fma_mixlo_f16 and v_fma_mixhi_f16, 7.8 ns, are what the compiler makes of one pair in four where the sums are not
// pinned: Q4_K's layer of 4096 tokens 439 us so, 429 pinned)
__device__ __forceinline__ uint32_t mix2(v2h u, float s, float c) {
    float lo = fmaf(float(u[0]), s, c), hi = fmaf(float(u[1]), s, c);
    asm("" : "+v"(lo), "+v"(hi));
    return bits_of(v2h{_Float16(lo), _Float16(hi)});
}
// bytes 0, 2 and bytes 1, 3 of u as halves 1024 + byte
__device__ __forceinline__ v2h bias_even(uint32_t u) { return as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04020400u)); }
__device__ __forceinline__ v2h bias_odd(uint32_t u) { return as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030401u)); }

// What the kernel needs of a format.
// kCodes: 1 KB transfers a bank and stage (64 lanes x 16 bytes): code() the lane's source, code_at() what to add
// for a transfer and stage. kRecs transfers for both banks' records: rec(), rec_at(). Prep: what decoding a stage needs in registers;
// slice(): piece j (16 bytes) of operand B; in items of up to kFold row tiles whole(), the piece without the super-block's factor fold(). kTab
// bytes of lookup table in LDS, filled by tables(). row_factors(): factors of whole weight rows.
template <uint32_t FMT> struct GroupedFormat;

struct GroupedWhole {                     // no factor outside the operands
    static constexpr int kFold = 0;
    template <class P> static __device__ __forceinline__ float fold(const P &) { return 1.f; }
    template <class P> static __device__ __forceinline__ uint4 whole(P &, int) { return uint4(); }
};
struct GroupedHalves : GroupedWhole {
    static constexpr bool kFp8 = false;
    static constexpr int kTab = 16;
    static __device__ __forceinline__ void tables(uint8_t *, int) {}
};
struct GroupedNibbles : GroupedHalves {   // 16 code bytes a sub-block in the canonical order
    static constexpr int kCodes = 1, kRecs = 1;
    static __device__ __forceinline__ const uint8_t * code(const BankView & b, int64_t tile, int S, int lane) { return b.codes + tile * S * 512 + lane * 16; }
    static __device__ __forceinline__ int code_at(int, int st) { return st * 1024; }
};

template <> struct GroupedFormat<TQMOE_IQ4_XS> : GroupedNibbles {
    static constexpr int kFold = 2;
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int, int lane) {
        const int l = lane & 31;   // sixteen lanes a bank; the upper half of the wave repeats the lower
        return (l < 16 ? b0.aux + tile0 * (S / 8) * 256 : b1.aux + tile1 * (S / 8) * 256) + (l & 15) * 16;
    }
    static __device__ __forceinline__ int rec_at(int, int st) { return (st >> 2) * 256; }
    struct Prep { uint32_t c[4]; float s, off, d; v2h ls, ls_off; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint8_t *, Prep & p) {
        const uint4 c = *reinterpret_cast<const uint4 *>(w + nb * 1024 + g * 512 + n * 16);
        const uint2 r = *reinterpret_cast<const uint2 *>(w + 2048 + nb * 256 + n * 8);
        p.c[0] = c.x; p.c[1] = c.y; p.c[2] = c.z; p.c[3] = c.w;
        p.d = half_bits_to_float(iq4xs_d_bits(r));
        const float ls = float(iq4xs_lsm32(r, (2 * st + g) & 7));
        p.s = p.d * ls;                // 17 bits: exact
        p.off = p.s * -1152.f;         // four more: exact
        p.ls = both(ls);
        p.ls_off = both(ls * -1152.f); // eight significant bits, at most 36864: exact
    }
    static __device__ __forceinline__ uint4 slice(Prep & p, int j) {
        return values(p, j, [&](v2h u) { return mix2(u, p.s, p.off); });
    }
    static __device__ __forceinline__ float fold(const Prep & p) { return p.d; }
    // value times the integer scale (up to 4064: rounded once, as the whole weight is in slice())
    static __device__ __forceinline__ uint4 whole(Prep & p, int j) {
        return values(p, j, [&](v2h u) { return bits_of(__builtin_elementwise_fma(u, p.ls, p.ls_off)); });
    }
    template <class F> static __device__ __forceinline__ uint4 values(const Prep & p, int j, F f) {
        constexpr Table16 t = table16({1, 24, 45, 63, 79, 93, 106, 118, 129, 141, 153, 166, 181, 197, 217, 241});   // the values + 128
        const uint32_t c = p.c[j], lo = pick(t, c & 0x0F0F0F0Fu), hi = pick(t, (c >> 4) & 0x0F0F0F0Fu);
        return make_uint4(f(bias_even(lo)), f(bias_odd(lo)), f(bias_even(hi)), f(bias_odd(hi)));
    }
};

template <> struct GroupedFormat<TQMOE_Q4_K> : GroupedNibbles {
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int, int lane) {
        return (lane < 32 ? b0.aux + tile0 * (S / 8) * 512 : b1.aux + tile1 * (S / 8) * 512) + (lane & 31) * 16;
    }
    static __device__ __forceinline__ int rec_at(int, int st) { return (st >> 2) * 512; }
    struct Prep { uint32_t c[4]; float s[2], off; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint8_t *, Prep & p) {
        const uint4 c = *reinterpret_cast<const uint4 *>(w + nb * 1024 + g * 512 + n * 16);
        const uint4 r = *reinterpret_cast<const uint4 *>(w + 2048 + nb * 512 + n * 16);
        p.c[0] = c.x; p.c[1] = c.y; p.c[2] = c.z; p.c[3] = c.w;
        // bytes (2 st + g) % 4 of the record's three dwords; the upper sub-blocks' six bits are a nibble and two top bits
        const bool upper = st & 2;
        const int sh = 16 * (st & 1) + 8 * g;
        const uint32_t low = upper ? 15u : 0u, six = upper ? 48u : 63u, from = upper ? 2u : 0u;
        const int sc = int(((r.w >> sh) & low) | ((r.y >> (sh + from)) & six)), mn = int(((r.w >> (sh + 4)) & low) | ((r.z >> (sh + from)) & six));
        const float s = half_bits_to_float(uint16_t(r.x & 0xFFFFu)) * float(sc);
        // A nibble alone in a half, in its low or the next four bits, is the subnormal number code * 2^-24 or 2^-20: the
        // multiply-add reads it as it is, and the scale takes the power of two (exact). (As the low bits of 1024 + code: an
        // instruction more a pair, and the constant that takes the bias off rounds; 4096 tokens 451 us so, 439 without.)
        p.s[0] = s * 0x1p24f;
        p.s[1] = s * 0x1p20f;
        p.off = -(half_bits_to_float(uint16_t(r.x >> 16)) * float(mn));
    }
    static __device__ __forceinline__ uint4 slice(Prep & p, int j) {
        const uint32_t c = p.c[j], c8 = c >> 8;
        auto low = [&](uint32_t x) { return mix2(as_h2(x & 0x000F000Fu), p.s[0], p.off); };
        auto high = [&](uint32_t x) { return mix2(as_h2(x & 0x00F000F0u), p.s[1], p.off); };
        return make_uint4(low(c), low(c8), high(c), high(c8));
    }
};

template <> struct GroupedFormat<TQMOE_Q6_K> : GroupedHalves {
    static constexpr int kFold = 2;
    static constexpr int kCodes = 1, kRecs = 3;   // low nibbles; then both banks' upper bits (512 bytes each) and each bank's records
    static __device__ __forceinline__ const uint8_t * code(const BankView & b, int64_t tile, int S, int lane) { return b.codes + tile * (S / 8) * 6144 + lane * 16; }
    static __device__ __forceinline__ int code_at(int, int st) { return (st >> 2) * 6144 + (st & 3) * 1024; }
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int i, int lane) {
        if (i == 0) return (lane < 32 ? b0.codes + tile0 * (S / 8) * 6144 : b1.codes + tile1 * (S / 8) * 6144) + 4096 + (lane & 31) * 16;
        return (i == 1 ? b0.aux + tile0 * (S / 8) * 1024 : b1.aux + tile1 * (S / 8) * 1024) + lane * 16;
    }
    static __device__ __forceinline__ int rec_at(int i, int st) { return i == 0 ? (st >> 2) * 6144 + (st & 3) * 512 : (st >> 2) * 1024; }
    struct Prep { uint32_t lo[4], hi[2]; float s[2], off[2], d; v2h sc[2], sc_off[2]; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint8_t *, Prep & p) {
        const uint4 c = *reinterpret_cast<const uint4 *>(w + nb * 1024 + g * 512 + n * 16);
        p.lo[0] = c.x; p.lo[1] = c.y; p.lo[2] = c.z; p.lo[3] = c.w;
        p.hi[0] = *reinterpret_cast<const uint32_t *>(w + 2048 + nb * 512 + n * 16 + g * 4);
        p.hi[1] = *reinterpret_cast<const uint32_t *>(w + 2048 + nb * 512 + n * 16 + 8 + g * 4);
        const uint8_t * r = w + 3072 + nb * 1024 + n * 32;
        const uint32_t s2 = *reinterpret_cast<const uint16_t *>(r + 2 * ((2 * st + g) & 7));
        p.d = half_bits_to_float(*reinterpret_cast<const uint16_t *>(r + 16));
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float sc = 0.25f * float(int(__builtin_amdgcn_sbfe(int(s2), 8 * i, 8)));   // the operand byte is four times the value
            p.s[i] = p.d * sc;
            p.off[i] = p.s[i] * -1152.f;           // 18 bits and four: exact
            p.sc[i] = both(sc);
            p.sc_off[i] = both(sc * -1152.f);      // eleven significant bits, at most 36864: exact
        }
    }
    static __device__ __forceinline__ float fold(const Prep & p) { return p.d; }
    static __device__ __forceinline__ uint4 slice(Prep & p, int j) {
        return values(p, j, [&](v2h u, int i) { return mix2(u, p.s[i], p.off[i]); });
    }
    // value times the integer scale (up to 4096: rounded once, as the whole weight is in slice())
    static __device__ __forceinline__ uint4 whole(Prep & p, int j) {
        return values(p, j, [&](v2h u, int i) { return bits_of(__builtin_elementwise_fma(u, p.sc[i], p.sc_off[i])); });
    }
    template <class F> static __device__ __forceinline__ uint4 values(const Prep & p, int j, F val) {
        // dword j of the low nibbles: half j / 2 of the sub-block, its operand dwords 2 (j % 2) and + 1
        const uint32_t lo = p.lo[j], hi = p.hi[j >> 1] >> (4 * (j & 1));
        const uint32_t a = ((lo << 2) & 0x3C3C3C3Cu) | ((hi << 6) & 0xC0C0C0C0u), b = ((lo >> 2) & 0x3C3C3C3Cu) | ((hi << 4) & 0xC0C0C0C0u);
        const uint32_t ua = a ^ 0x80808080u, ub = b ^ 0x80808080u;
        return make_uint4(val(bias_even(ua), 0), val(bias_odd(ua), 0), val(bias_even(ub), 1), val(bias_odd(ub), 1));
    }
};

template <> struct GroupedFormat<TQMOE_IQ3_S> : GroupedHalves {
    static constexpr int kFold = 1;
    // Points 0..255 are the table's first 2 KB; the others follow 2 and again 4 KB behind it, so that an index's ninth bit is an
    // address bit after one shift for two of them.
    static constexpr int kCodes = 1, kRecs = 1, kTab = 6144;
    static __device__ __forceinline__ void tables(uint8_t * tab, int tid) {   // a lattice point's magnitudes as halves, weights 0, 2, 1, 3
        for (int i = tid; i < 512; i += 256) {
            const v2h bias = as_h2(0xE400E400u);       // -1024
            const uint32_t m = d_iq3s_grid.v[i];
            const uint2 v = make_uint2(bits_of(bias_even(m) + bias), bits_of(bias_odd(m) + bias));
            if (i < 256) reinterpret_cast<uint2 *>(tab)[i] = v;
            else {
#pragma unroll
                for (int c = 1; c <= 2; ++c) reinterpret_cast<uint2 *>(tab)[c * 256 + i - 256] = v;
            }
        }
    }
    static __device__ __forceinline__ const uint8_t * code(const BankView & b, int64_t tile, int S, int lane) {   // the pair's indices, then the signs
        return b.codes + tile * (S / 8) * 3072 + (lane < 32 ? 0 : 2048) + (lane & 31) * 16;
    }
    // (indices: 512 bytes a pair, signs: 512 bytes two pairs; the lane's own step)
    static __device__ __forceinline__ int code_at(int, int st) { return (st >> 2) * 3072 + ((threadIdx.x & 32) ? ((st & 3) >> 1) * 512 : (st & 3) * 512); }
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int, int lane) {
        return (lane < 32 ? b0.aux + tile0 * (S / 8) * 512 : b1.aux + tile1 * (S / 8) * 512) + (lane & 31) * 16;
    }
    static __device__ __forceinline__ int rec_at(int, int st) { return (st >> 2) * 512; }
    struct Prep { uint32_t qs[2], sg, qh; v2h sc, d; const uint8_t * lat; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int st, int n, int g, const uint8_t * tab, Prep & p) {
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
        p.lat = tab;
    }
    static __device__ __forceinline__ float fold(const Prep & p) { return float(p.d[0]); }
    static __device__ __forceinline__ uint4 slice(Prep & p, int j) { return values<true>(p, j); }
    static __device__ __forceinline__ uint4 whole(Prep & p, int j) { return values<false>(p, j); }
    template <bool D> static __device__ __forceinline__ uint4 values(const Prep & p, int j) {
        const int h = j >> 1, q = 2 * (j & 1);     // operand dwords q and q + 1 of half h: weights 4 j .. and 16 + 4 j ..
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int s = 4 * h + q + i;           // bit 8 t + s: the sign of weight t
            uint32_t at = ((p.qs[h] >> (8 * (q + i))) & 0xFFu) << 3;   // (a byte shifted: one instruction, where nothing is merged into it)
            asm("" : "+v"(at));
            const uint2 mag = *reinterpret_cast<const uint2 *>(p.lat + (at | ((p.qh << (11 - (s & 6))) & (0x800u << (s & 1)))));   // the four magnitudes as halves, weights 0, 2 and 1, 3
            // times the integer scale (exact), times d (the one rounding)
            v2h a = as_h2(mag.x ^ ((p.sg << (15 - s)) & 0x80008000u)) * p.sc, b = as_h2(mag.y ^ ((p.sg << (7 - s)) & 0x80008000u)) * p.sc;
            if constexpr (D) { a *= p.d; b *= p.d; }
            v[2 * i] = bits_of(a);
            v[2 * i + 1] = bits_of(b);
        }
        return make_uint4(v[0], v[1], v[2], v[3]);
    }
};

template <> struct GroupedFormat<TQMOE_NVFP4G> : GroupedWhole {
    static constexpr bool kFp8 = true;
    static constexpr int kCodes = 2, kRecs = 1, kTab = 256 * 8;
    // Per scale byte the products e2m1(code) * e4m3(scale) / 8 of the eight codes without a sign, rounded to E4M3 (nearest even; an
    // eighth keeps the largest, 6 * 448, inside the format, row_factors gives it back): rounding knows no sign, so that a code's own is
    // bit 7 of the result.
    static __device__ __forceinline__ void tables(uint8_t * tab, int tid) {
        const float sc = e4m3_to_float(uint32_t(tid));
        uint32_t v[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            float f[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = float(((q == 0 ? kFp4T0 : kFp4T1) >> (8 * j)) & 0xFFu) * 0.0625f * sc;
            const int w = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
            v[q] = uint32_t(__builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w, true));
        }
        const bool none = (tid & 0x7F) == 0x7F;   // (not a number, in E4M3 too)
        reinterpret_cast<uint2 *>(tab)[tid] = none ? make_uint2(0x7F7F7F7Fu, 0x7F7F7F7Fu) : make_uint2(v[0], v[1]);
    }
    // The products of the low (high) nibbles of four code bytes: four instructions, where a table of sixteen takes five and six (with the row
    // factors read once an item, 8192 tokens of 8 of 256 experts 1642 -> 1464 us a layer, products 1430 -> 1281).
    static __device__ __forceinline__ uint32_t low4(uint2 t, uint32_t c) { return __builtin_amdgcn_perm(t.y, t.x, c & 0x07070707u) ^ ((c << 4) & 0x80808080u); }
    static __device__ __forceinline__ uint32_t high4(uint2 t, uint32_t c) { return __builtin_amdgcn_perm(t.y, t.x, (c >> 4) & 0x07070707u) ^ (c & 0x80808080u); }
    static __device__ __forceinline__ const uint8_t * code(const BankView & b, int64_t tile, int S, int lane) { return b.codes + tile * S * 512 + lane * 16; }
    static __device__ __forceinline__ int code_at(int i, int st) { return st * 2048 + i * 1024; }
    static __device__ __forceinline__ const uint8_t * rec(const BankView & b0, const BankView & b1, int64_t tile0, int64_t tile1, int S, int, int lane) {
        const int l = lane & 31;   // eight bytes a row and stage: sixteen lanes a bank, the upper half of the wave repeats the lower
        return (l < 16 ? b0.aux + tile0 * (S / 4) * 256 : b1.aux + tile1 * (S / 4) * 256) + (l & 15) * 16;
    }
    static __device__ __forceinline__ int rec_at(int, int st) { return st * 256; }
    struct Prep { uint32_t c[2][4], sc[2]; uint2 t0, t1; const uint8_t * tab; };
    static __device__ __forceinline__ void prep(const uint8_t * w, int nb, int, int n, int g, const uint8_t * tab, Prep & p) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {   // sub-blocks g and 2 + g
            const uint4 c = *reinterpret_cast<const uint4 *>(w + nb * 2048 + i * 1024 + g * 512 + n * 16);
            p.c[i][0] = c.x; p.c[i][1] = c.y; p.c[i][2] = c.z; p.c[i][3] = c.w;
        }
        const uint2 r = *reinterpret_cast<const uint2 *>(w + 4096 + nb * 256 + n * 8);
        p.sc[0] = r.x >> (16 * g);
        p.sc[1] = r.y >> (16 * g);
        p.tab = tab;
    }
    static __device__ __forceinline__ uint4 slice(Prep & p, int j) {
        const int i = j >> 1, h = j & 1;
        if (h == 0) {
            p.t0 = *reinterpret_cast<const uint2 *>(p.tab + (p.sc[i] & 0xFFu) * 8);
            p.t1 = *reinterpret_cast<const uint2 *>(p.tab + ((p.sc[i] >> 8) & 0xFFu) * 8);
        }
        const uint32_t a = p.c[i][2 * h], b = p.c[i][2 * h + 1];
        return make_uint4(low4(p.t0, a), high4(p.t1, a), low4(p.t0, b), high4(p.t1, b));
    }
    static __device__ __forceinline__ void row_factors(const BankView & b, int64_t row, float * f) {   // of four rows
        const float4 v = *reinterpret_cast<const float4 *>(b.aux + nvfp4_global_offset(b.rows_total, b.cols) + row * 4);
        f[0] = 8.f * v.x; f[1] = 8.f * v.y; f[2] = 8.f * v.z; f[3] = 8.f * v.w;
    }
};

template <bool PIN> __device__ __forceinline__ uint32_t half_pair(float x, float y) {
    if constexpr (PIN) asm("" : "+v"(x), "+v"(y));   // (the product is rounded before it is converted)
    return bits_of(v2h{_Float16(x), _Float16(y)});
}

// bytes of a wave's codes and records of one stage
template <class W> constexpr int kStageW = 2 * W::kCodes * 1024 + W::kRecs * 1024;
template <class W> constexpr int kStageCols = W::kFp8 ? 128 : 64;   // columns of a stage: 128 bytes of a row
// blocks a compute unit holds (four waves each, so waves a SIMD): the accumulators of MAX row tiles set the registers
template <class W, int MAX> constexpr int kGroupedWaves = MAX == 4 || (MAX == 2 && W::kFold == 2) ? 2 : 3;
// Stages of input rows and of codes in LDS for MT row tiles, in the part of a compute unit's 160 KB that one of its blocks may
// take. Codes come from HBM and may be two and more stages on their way; rows come from the L2 (an item's other blocks read
// the same). (Q4_K at 4096 tokens: 554 us a layer with one stage of codes under way, 521 with two.) With three blocks a unit
// their own turns hide the trip, and two stages are the faster ring (three / two, us a layer, items of 64 rows: IQ3_S, 512 tokens of 8 experts
// of 256 215 / 211, IQ4_XS, 333 skewed tokens 127.5 / 125.6, Q4_K, 200 tokens of 64 experts 83.2 / 82.4); with two blocks two
// to five are the same to 0.5 %.
template <class W, int MT, int MAX> struct Rings {
    static constexpr int kLds = 163840 / kGroupedWaves<W, MAX> - W::kTab - 1280;   // what one of the unit's blocks may take
    static constexpr int kRows = MT == 4 || kGroupedWaves<W, MAX> == 3 ? 2 : MT == 2 || kStageW<W> > 4096 ? 3 : 4;
    static constexpr int kRoom = (kLds - kRows * MT * 4096) / (4 * kStageW<W>);
    static constexpr int kMost = kGroupedWaves<W, MAX> == 3 ? 2 : 5, kCodes = kRoom < kMost ? kRoom : kMost;
    static_assert(kCodes >= 2, "two stages of codes");
    static constexpr int kBytes = kRows * MT * 4096 + 4 * kCodes * kStageW<W>;
};
template <class W, int MAX> constexpr int grouped_lds() {
    const int a = Rings<W, 1, MAX>::kBytes, b = Rings<W, MAX == 4 ? 2 : MAX, MAX>::kBytes, c = Rings<W, MAX, MAX>::kBytes;
    return a > b ? (a > c ? a : c) : (b > c ? b : c);
}

template <uint32_t FMT, int MAX, bool GATEUP, class OT>   // MAX: row tiles of an item at most
__global__ __launch_bounds__(256, (kGroupedWaves<GroupedFormat<FMT>, MAX>)) void grouped_rows_k(GroupedArgs k) {
    using W = GroupedFormat<FMT>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];   // [kRows][MT * 4096] input rows | [4 waves][kCodes][kStageW] codes and records
    __shared__ __attribute__((aligned(16))) uint8_t s_tab[W::kTab];
    constexpr int kItemRows = 32 * MAX;
    __shared__ int s_asg[kItemRows];
    __shared__ float s_scale[kItemRows];
    // An item's groups of weight tiles run on one XCD one after the other (its rows stay in that L2), and an XCD takes a run
    // of consecutive items, an expert's items among them, of every class (its weights do too): see grouped_plan_k.
    const int xcd = int(blockIdx.x) & 7, at = int(blockIdx.x) >> 3, grp = at % k.groups;
    const int4 counts = k.plan[0];
    int slot = at / k.groups, base = 0, chunk = -1;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int items = c == 0 ? counts.x : c == 1 ? counts.y : c == 2 ? counts.z : counts.w, per = (items + 7) >> 3;
        if (chunk < 0 && slot < per) {
            if (xcd * per + slot >= items) return;
            chunk = base + xcd * per + slot;
        }
        slot -= per;
        base += items;
    }
    if (chunk < 0) return;
    const int4 item = k.plan[1 + chunk];           // expert, its first row in perm, rows, first row tile
    const int e = item.x, cnt = item.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 31, g = lane >> 5;
    const int rows = k.b0.rows, cols = k.b0.cols, S = cols / 32, tiles = rows / 32;
    const bool is_shared = e == k.shared_expert;
    const int row_lim = GATEUP && is_shared ? k.shared_lim : rows;
    const int stages = (!GATEUP && is_shared ? k.shared_lim : cols) / kStageCols<W>;
    W::tables(s_tab, tid);
    if (tid < kItemRows) {
        s_asg[tid] = tid < cnt ? k.perm[item.y + tid] : -1;
        s_scale[tid] = 1.f;
        if (k.xs && tid < cnt) s_scale[tid] = k.xs[W::kFp8 && k.row_tiles ? item.w * 32 + tid : s_asg[tid] / k.xdiv];
    }
    __syncthreads();
    // weight tiles of this wave (past the last one: it once more, not stored)
    int wt[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) wt[b] = GATEUP ? grp * 4 + wave : grp * 8 + wave * 2 + b;

    auto body = [&](auto tag) {
        constexpr int MT = decltype(tag)::value;
        constexpr bool FOLD = MAX <= W::kFold;
        v16f acc[2][MT];
        [[maybe_unused]] v16f part[2][FOLD ? MT : 1];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[b][m][i] = 0.f;
        if constexpr (FOLD)
#pragma unroll
            for (int m = 0; m < MT; ++m) part[0][m] = part[1][m] = acc[0][0];
        const bool any = GATEUP ? grp * 128 < row_lim : true;
        if (any) {
            using R = Rings<W, MT, MAX>;
            constexpr int LA = R::kRows - 1, LW = R::kCodes, LM = LA > LW ? LA : LW;   // stages ahead: stage t sends the rows of t + LA and the codes of t + LW
            constexpr int NA = MT, NW = 2 * W::kCodes + W::kRecs;   // transfers a wave sends for a stage
            // input rows: transfer q of a wave is rows 8 (4 q + wave) .. + 7 of the stage's 128 bytes, a row's piece p in slot
            // p ^ (row / 2 & 7): the operand reads (a row a lane) then find sixteen rows' pieces in the sixteen 16-byte groups of
            // the 64 banks (rows are half as long as a line of banks)
            const uint8_t * a_src[MT];
#pragma unroll
            for (int q = 0; q < MT; ++q) {
                const int row = (4 * q + wave) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
                if (W::kFp8 && k.row_tiles)   // operand-major tiles of 32 rows: 1 KB a sub-block, the rows' first halves, then their second
                    a_src[q] = static_cast<const uint8_t *>(k.x) + (int64_t(item.w) + (row >> 5)) * 32 * cols + (piece >> 1) * 1024 + (piece & 1) * 512 + (row & 31) * 16;
                else
                    a_src[q] = static_cast<const uint8_t *>(k.x) + (int64_t(max(s_asg[row], 0)) / k.xdiv * cols) * (W::kFp8 ? 1 : 2) + piece * 16;
            }
            const int a_step = W::kFp8 && k.row_tiles ? 4096 : 128;
            const uint32_t lds0 = lds_address(lds);
            uint8_t * const w_lds = lds + R::kRows * MT * 4096 + wave * R::kCodes * kStageW<W>;
            const uint32_t w_lds0 = lds_address(w_lds);
            const int64_t t0 = int64_t(e) * tiles + min(wt[0], tiles - 1), t1 = int64_t(e) * tiles + min(wt[1], tiles - 1);
            const uint8_t * c_src[2] = {W::code(k.b0, t0, S, lane), W::code(k.b1, t1, S, lane)}, * r_src[W::kRecs];
#pragma unroll
            for (int i = 0; i < W::kRecs; ++i) r_src[i] = W::rec(k.b0, k.b1, t0, t1, S, i, lane);
            auto send_a = [&](int st, int slot) {
                if (st >= stages) return;
#pragma unroll
                for (int q = 0; q < MT; ++q) dma16(a_src[q] + st * a_step, lds0 + slot * MT * 4096 + (4 * q + wave) * 1024);
            };
            auto send_w = [&](int st, int slot) {
                if (st >= stages) return;
                const uint32_t to = w_lds0 + slot * kStageW<W>;
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < W::kCodes; ++i) dma16(c_src[b] + W::code_at(i, st), to + (b * W::kCodes + i) * 1024);
#pragma unroll
                for (int i = 0; i < W::kRecs; ++i) dma16(r_src[i] + W::rec_at(i, st), to + (2 * W::kCodes + i) * 1024);
            };
            const uint8_t * a_row = lds + n * 128;
            uint4 bw[2][4];
            typename W::Prep pr[2];
            auto operand = [&](typename W::Prep & p, int j) {
                if constexpr (FOLD) return W::whole(p, j);
                else return W::slice(p, j);
            };
#pragma unroll
            for (int t = -LM; t < 0; ++t) {   // what the stages before the first would have sent
                if (t + LA >= 0) send_a(t + LA, t + LA);
                if (t + LW >= 0) send_w(t + LW, t + LW);
            }
            if (LM <= stages) dma_wait<(LW - 1) * NW + (LA < LW ? LA : LW - 1) * NA, false>(); else dma_wait<0, false>();
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                W::prep(w_lds, b, 0, n, g, s_tab, pr[b]);
#pragma unroll
                for (int j = 0; j < 4; ++j) bw[b][j] = operand(pr[b], j);
            }
            int a_at = 0, w_at = 0;           // slots of this stage's rows and codes
            for (int st = 0; st < stages; ++st) {
                // this stage's rows and the next one's codes are here (what the stages since have sent may be under way, where
                // they have sent all), and every wave is done with the slots that are filled now
                constexpr int kSinceA = NW + (LA - 1) * (NA + NW), kSinceW = (LW - 2) * (NA + NW);
                if (st + LM <= stages) dma_wait<(kSinceA < kSinceW ? kSinceA : kSinceW), true>(); else dma_wait<0, true>();
                send_a(st + LA, a_at == 0 ? LA : a_at - 1);
                send_w(st + LW, w_at);
                w_at = w_at + 1 == LW ? 0 : w_at + 1;
                const bool more = st + 1 < stages;   // (past the last stage: its own codes again, not used)
                const int w_next = more ? w_at : w_at == 0 ? LW - 1 : w_at - 1;
                float d[2];
                if constexpr (FOLD) {
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        d[b] = W::fold(pr[b]);
                        asm("" : "+v"(d[b]));      // (in fp32: a mixed multiply-add takes half as long again)
                    }
                }
#pragma unroll
                for (int b = 0; b < 2; ++b) W::prep(w_lds + w_next * kStageW<W>, b, more ? st + 1 : st, n, g, s_tab, pr[b]);
                const uint8_t * a_buf = a_row + a_at * MT * 4096;
                a_at = a_at + 1 == LA + 1 ? 0 : a_at + 1;
                uint4 a[2][MT];
                // piece j of a row is the 16 bytes that go with piece j of operand B (E4M3: two pieces are one operand)
                auto read_a = [&](int j) {
                    const int piece = W::kFp8 ? 4 * (j >> 1) + 2 * g + (j & 1) : 4 * g + j;
#pragma unroll
                    for (int m = 0; m < MT; ++m) a[j & 1][m] = *reinterpret_cast<const uint4 *>(a_buf + m * 4096 + ((piece ^ ((n >> 1) & 7)) * 16));
                };
                read_a(0);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (W::kFp8) {
                        if (j & 1) continue;
                        read_a(j + 1);
#pragma unroll
                        for (int b = 0; b < 2; ++b)
#pragma unroll
                            for (int m = 0; m < MT; ++m)
                                acc[b][m] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(join(bw[b][j], bw[b][j + 1]), join(a[0][m], a[1][m]), acc[b][m], 0, 0, 0, 0, 0, 0);
                        if (j < 2) read_a(j + 2);
#pragma unroll
                        for (int b = 0; b < 2; ++b) { bw[b][j] = W::slice(pr[b], j); bw[b][j + 1] = W::slice(pr[b], j + 1); }
                    } else {
                        if (j < 3) read_a(j + 1);
#pragma unroll
                        for (int b = 0; b < 2; ++b)
#pragma unroll
                            for (int m = 0; m < MT; ++m) {
                                if constexpr (FOLD) part[b][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[j & 1][m]), __builtin_bit_cast(v8h, bw[b][j]), part[b][m], 0, 0, 0);
                                else acc[b][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, bw[b][j]), __builtin_bit_cast(v8h, a[j & 1][m]), acc[b][m], 0, 0, 0);
                            }
#pragma unroll
                        for (int b = 0; b < 2; ++b) bw[b][j] = operand(pr[b], j);
                    }
                }
                if constexpr (FOLD) {
                    if ((st & 3) == 3 || !more) {
#pragma unroll
                        for (int b = 0; b < 2; ++b)
#pragma unroll
                            for (int m = 0; m < MT; ++m)
#pragma unroll
                                for (int i = 0; i < 16; ++i) {
                                    acc[b][m][i] = fmaf(part[b][m][i], d[b], acc[b][m][i]);
                                    part[b][m][i] = 0.f;
                                }
                    }
                }
            }
        }
        // The weights are the first operand: result register 4 c + i of lane (n, g) is weight row 8 c + 4 g + i of the tile and
        // input row n of the row tile: a lane has four consecutive values of one row at a time. They go through the wave's own
        // LDS (its codes are done with) and leave as 16 bytes a lane, a row's 64 or 128 bytes together.
        constexpr int kPitch = 32 * sizeof(OT) + 16, kLanes = 32 * sizeof(OT) / 16, kStep = 64 / kLanes;   // lanes a row, rows a store
        static_assert(32 * kPitch <= Rings<W, MT, MAX>::kCodes * kStageW<W>, "the tile's place");
        uint8_t * const tile_lds = lds + Rings<W, MT, MAX>::kRows * MT * 4096 + wave * Rings<W, MT, MAX>::kCodes * kStageW<W>;
        [[maybe_unused]] float own[2][W::kFp8 ? 16 : 1];   // (read once: between an item's stores every read would wait for the memory)
        if constexpr (W::kFp8)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int c = 0; c < 4; ++c) W::row_factors(b ? k.b1 : k.b0, (int64_t(e) * tiles + min(wt[b], tiles - 1)) * 32 + 8 * c + 4 * g, &own[b][4 * c]);
        const bool clamp = k.glu.limit > 1e-6f;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float scl = s_scale[m * 32 + n];
#pragma unroll
            for (int b = 0; b < (GATEUP ? 1 : 2); ++b) {
                if (wt[b] >= tiles) continue;
                auto factors = [&](int bank, float (&v)[16]) {   // the weight rows' own factors, the input row's scale
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        v[i] = acc[bank][m][i];
                        if constexpr (W::kFp8) v[i] *= own[bank][i];
                        v[i] *= FOLD ? s_scale[m * 32 + 8 * (i >> 2) + 4 * g + (i & 3)] : scl;
                    }
                };
                float v[16];
                factors(b, v);
                if constexpr (GATEUP) {
                    float u[16];
                    factors(1, u);
                    if (clamp) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) glu_clamp_inputs(k.glu, v[i], u[i]);
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[i] *= __builtin_amdgcn_rcpf(1.f + __expf(-v[i]));
                    if (clamp) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) v[i] = glu_clamp_silu(k.glu, v[i]);
                    }
                    const bool live = wt[0] * 32 < row_lim;   // (zeros past the shared expert's rows, whatever the bank holds there)
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[i] = live ? v[i] * u[i] : 0.f;
                }
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float * q = v + 4 * c;
                    uint8_t * to = tile_lds + n * kPitch;
                    if constexpr (FOLD) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            uint8_t * row = tile_lds + (8 * c + 4 * g + i) * kPitch;
                            if constexpr (sizeof(OT) == 4) reinterpret_cast<float *>(row)[n] = q[i];
                            else reinterpret_cast<_Float16 *>(row)[GATEUP ? operand_pos(n) : n] = _Float16(q[i]);
                        }
                    } else if constexpr (sizeof(OT) == 4) *reinterpret_cast<float4 *>(to + (8 * c + 4 * g) * 4) = make_float4(q[0], q[1], q[2], q[3]);
                    else if constexpr (GATEUP && !W::kFp8)   // operand_pos: the four values stay together, 1 and 2 change places
                        *reinterpret_cast<uint2 *>(to + operand_pos(8 * c + 4 * g) * 2) = make_uint2(half_pair<W::kFp8>(q[0], q[2]), half_pair<W::kFp8>(q[1], q[3]));
                    else *reinterpret_cast<uint2 *>(to + (8 * c + 4 * g) * 2) = make_uint2(half_pair<W::kFp8>(q[0], q[1]), half_pair<W::kFp8>(q[2], q[3]));
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int q = 0; q < 32 / kStep; ++q) {
                    const int row = q * kStep + lane / kLanes, asg = s_asg[m * 32 + row];
                    const uint4 w = *reinterpret_cast<const uint4 *>(tile_lds + row * kPitch + (lane % kLanes) * 16);
                    if (asg >= 0) *reinterpret_cast<uint4 *>(static_cast<OT *>(k.out) + int64_t(asg) * rows + wt[b] * 32 + (lane % kLanes) * (16 / sizeof(OT))) = w;
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
    };
    if (MAX == 1 || cnt <= 32) body(std::integral_constant<int, 1>{});
    else if (MAX == 2 || cnt <= 64) body(std::integral_constant<int, MAX == 1 ? 1 : 2>{});
    else body(std::integral_constant<int, MAX>{});
}

template <uint32_t FMT, int MAX> void grouped_rows_launch_max(const GroupedArgs & k, bool gateup, bool f32_out, unsigned blocks, hipStream_t s) {
    constexpr int bytes = grouped_lds<GroupedFormat<FMT>, MAX>();
    auto go = [&](auto kernel) {
        allow_dynamic_lds(reinterpret_cast<const void *>(kernel), bytes);
        kernel<<<blocks, 256, bytes, s>>>(k);
    };
    if (gateup) {
        if constexpr (MAX > 1 || GroupedFormat<FMT>::kFold) go(&grouped_rows_k<FMT, MAX, true, uint16_t>);   // (grouped_rows_per_item)
    } else if (f32_out) go(&grouped_rows_k<FMT, MAX, false, float>);
    else go(&grouped_rows_k<FMT, MAX, false, uint16_t>);
}
template <uint32_t FMT> void grouped_rows_launch(const GroupedArgs & k, int item_rows, bool gateup, bool f32_out, unsigned blocks, hipStream_t s) {
    if constexpr (!GroupedFormat<FMT>::kFp8) {
        if (item_rows == 32) return grouped_rows_launch_max<FMT, 1>(k, gateup, f32_out, blocks, s);
        if (item_rows == 64) return grouped_rows_launch_max<FMT, 2>(k, gateup, f32_out, blocks, s);
    }
    grouped_rows_launch_max<FMT, 4>(k, gateup, f32_out, blocks, s);
}

}  // namespace
}  // namespace tqmoe
