// Grouped int8 products on rows that lie as the quantiser left them (a row per token or per assignment), one operand plane a weight.
//
// A block of four waves takes one item of the plan (an expert and up to 32 or 64 of its input rows) and eight tiles of 32 weight
// rows, two a wave: the same tile of the gate and the up bank, or two tiles of one bank. Per stage (128 columns: four sub-blocks):
//  * the rows go through registers into LDS a stage ahead, one barrier a stage; no gathered copy of them exists;
//  * a lane loads eight code bytes of its weight row and sub-block a stage ahead, straight into registers (coalesced: the banks are
//    tile-major), and turns them into the sixteen int8 table values that are its operand, 44 vector instructions;
//  * one v_mfma_i32_32x32x32_i8 a (row tile, weight tile, sub-block): its sixteen sums a lane are scaled while the next
//    unit's product runs. A lane has one weight row, so that the weights' scales need no exchange.
// The scale of a sub-block is applied to the sums and not inside the operand (where the 13-bit product of value and scale takes two
// planes, two products and twice the look-ups): rows with one scale: a 24-bit integer multiply-add into the super-block's integer sum,
// one fp32 multiply-add a super-block; rows with a scale per 32 values: sums to fp32, times the weight's scale (one multiply-add for
// both), times the row's into the fp32 result. Order and roundings are those of plane_gemm_k: equal bits.
//
// Bound by vector instructions: a unit (65,536 operations) is one product (32 cycles of the matrix pipe, about 18 of the
// vector issue) and 16 multiply-adds and 4 folds of 4 to 5 cycles each (a scale per 32 values: 32), the operand's decode (22) spread over
// the item's row tiles. 4096 tokens of 10 of 512 experts, Zipf, in the kernel trace: gate / up 342 us on plane_gemm_k, 269 here (vector pipe
// 80 % active, matrix pipe 16 %), down 231 and 161, and the two launches that gathered rows (55 us) are one that quantises them (17); with a
// scale per 32 values gate / up 589 and 328 us (vector pipe 99 %), down 357 and 198, no launch between (a weight tile's act values are one block of 32: the gate / up product quantises them itself).
#pragma once
#include "decode_table.cuh"
#include "formats.cuh"
#include "grouped_rows_api.cuh"
#include "int8_fold.cuh"
#include "row_quant.cuh"

namespace tqmoe {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

template <uint32_t FMT> struct Int8Format;

template <> struct Int8Format<TQMOE_IQ4_XS> {
    typedef uint2 Code;   // eight code bytes of a sub-block: sixteen weights
    typedef uint2 Rec;
    static __device__ __forceinline__ const uint8_t * codes(const BankView & b, int64_t tile, int S) { return b.codes + tile * S * 512; }
    static __device__ __forceinline__ const uint8_t * recs(const BankView & b, int64_t tile, int S) { return b.aux + tile * (S / 8) * 256; }
    static __device__ __forceinline__ Code code(const uint8_t * p, int sub, int n, int g) { return *reinterpret_cast<const uint2 *>(p + sub * 512 + n * 16 + g * 8); }
    static __device__ __forceinline__ Rec rec(const uint8_t * p, int sb, int n) { return *reinterpret_cast<const uint2 *>(p + sb * 256 + n * 8); }
    static __device__ __forceinline__ v4i operand(Code c) {
        constexpr Table16 t = table16({-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113});
        const uint32_t m = 0x0F0F0F0Fu;
        return v4i{int(pick(t, c.x & m)), int(pick(t, (c.x >> 4) & m)), int(pick(t, c.y & m)), int(pick(t, (c.y >> 4) & m))};
    }
    static __device__ __forceinline__ int scale(const Rec & r, int ib) { return iq4xs_lsm32(r, ib); }
    static __device__ __forceinline__ float d(const Rec & r) { return half_bits_to_float(iq4xs_d_bits(r)); }
};

// MAX: row tiles of an item at most. BLK: the rows carry a scale per 32 values (k.xs: [rows][cols / 32]), else one a row.
// BLK and GATEUP: the act rows leave as int8 with a scale per 32 values (k.out, k.out_scale), else results are halves.
template <uint32_t FMT, bool BLK, int MAX, bool GATEUP>
__global__ __launch_bounds__(256, MAX == 1 ? 3 : 2) void grouped_i8_k(GroupedArgs k) {
    using W = Int8Format<FMT>;
    constexpr int kItemRows = 32 * MAX;
    constexpr int kOutCols = GATEUP ? 32 : 64, kPitch = kOutCols * 2 + 16;
    __shared__ __attribute__((aligned(16))) uint8_t s_rows[2][MAX * 4096];      // [row][128 bytes], a row's piece p in slot p ^ (row / 2 & 7)
    __shared__ __attribute__((aligned(16))) float s_bs[BLK ? 2 : 1][BLK ? MAX * 128 : 4];   // [row tile][sub-block][32 rows]
    __shared__ __attribute__((aligned(16))) uint8_t s_out[4][32 * kPitch];
    __shared__ int s_asg[kItemRows], s_row[kItemRows];   // assignments, their input rows
    __shared__ __attribute__((aligned(16))) float s_scale[kItemRows];
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
    const int e = __builtin_amdgcn_readfirstlane(item.x), cnt = __builtin_amdgcn_readfirstlane(item.z);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 31, g = lane >> 5;
    const int rows = k.b0.rows, cols = k.b0.cols, S = cols / 32, tiles = rows / 32;
    const bool is_shared = e == k.shared_expert;
    const int row_lim = GATEUP && is_shared ? k.shared_lim : rows;
    const int NSB = (!GATEUP && is_shared ? k.shared_lim : cols) / 256, stages = 2 * NSB;
    if (tid < kItemRows) {
        const int asg = tid < cnt ? k.perm[item.y + tid] : -1, row = max(asg, 0) / k.xdiv;
        s_asg[tid] = asg;
        s_row[tid] = row;
        s_scale[tid] = !BLK && tid < cnt ? k.xs[row] : 1.f;
    }
    __syncthreads();
    int wt[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) wt[b] = GATEUP ? grp * 4 + wave : grp * 8 + wave * 2 + b;

    auto body = [&](auto tag) {
        constexpr int MT = decltype(tag)::value;
        float acc[2][MT][16];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[b][m][i] = 0.f;
        if (GATEUP ? grp * 128 < row_lim : true) {
            // Where sums go to fp32 one by one, a product starts from the bits of kBias = 1.5 * 2^23: its result p, read as a float, is
            // kBias + p (|p| is at most 32 * 127 * 127), and one multiply-add to kBias * -d, which is exact (d has 17 bits), is p * d rounded
            // once, as conversion and multiplication give it. (us a layer of 512 experts, converted / from the bits: 64 tokens 229 / 202, 1501
            // 383 / 356, 8192 1302 / 1182.)
            constexpr float kBias = 12582912.f;
            v16i start;
#pragma unroll
            for (int i = 0; i < 16; ++i) start[i] = BLK ? __builtin_bit_cast(int, kBias) : 0;
            if constexpr (BLK) asm volatile("" : "+v"(start));   // (sixteen registers kept; they would be written for every product)
            int isum[2][MT][BLK ? 1 : 16];
            const uint8_t * x_src[MT];
            const float * s_src = nullptr;
#pragma unroll
            for (int m = 0; m < MT; ++m) x_src[m] = static_cast<const uint8_t *>(k.x) + int64_t(s_row[m * 32 + (tid >> 3)]) * cols + (tid & 7) * 16;
            const int s_tile = MT == 2 ? tid >> 7 : 0;
            if constexpr (BLK) s_src = k.xs + int64_t(s_row[s_tile * 32 + (tid & 31)]) * S + ((tid >> 5) & 3);
            const uint8_t * c_src[2], * r_src[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int64_t t = int64_t(e) * tiles + min(wt[b], tiles - 1);
                c_src[b] = W::codes(b ? k.b1 : k.b0, t, S);
                r_src[b] = W::recs(b ? k.b1 : k.b0, t, S);
            }
            uint4 xr0, xr1;   // (an array would be placed in scratch memory)
            float sr = 0.f;
            auto load_rows = [&](int st) {
                st = min(st, stages - 1);
                xr0 = *reinterpret_cast<const uint4 *>(x_src[0] + st * 128);
                if constexpr (MT == 2) xr1 = *reinterpret_cast<const uint4 *>(x_src[1] + st * 128);
                if constexpr (BLK) sr = s_src[st * 4];
            };
            auto put_rows = [&](int buf) {
                const int row = tid >> 3;
                uint8_t * to = &s_rows[buf][row * 128 + (((tid & 7) ^ ((row >> 1) & 7)) * 16)];
                *reinterpret_cast<uint4 *>(to) = xr0;
                if constexpr (MT == 2) *reinterpret_cast<uint4 *>(to + 4096) = xr1;
                if constexpr (BLK) s_bs[buf][s_tile * 128 + (tid & 127)] = sr;
            };
            typename W::Code code[2][4];
            typename W::Rec rec[2], rec_next[2];
            load_rows(0);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                rec_next[b] = W::rec(r_src[b], 0, n);
#pragma unroll
                for (int i = 0; i < 4; ++i) code[b][i] = W::code(c_src[b], i, n, g);
            }
            put_rows(0);
            load_rows(1);
            for (int sb = 0; sb < NSB; ++sb) {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    rec[b] = rec_next[b];
                    rec_next[b] = W::rec(r_src[b], min(sb + 1, NSB - 1), n);
                }
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int st = 2 * sb + half, st_next = min(st + 1, stages - 1);
                    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    put_rows(1 - half);
                    load_rows(st + 2);
                    constexpr bool kLate = BLK && MAX == 1;   // one set of sums and of the rows' scales: three waves a SIMD have no registers for two (31 spilled, 1501 tokens 378 -> 432)
                    v16i pend;
                    [[maybe_unused]] float4 pend_s[4];
                    auto fold = [&](int u) {   // unit u of the stage: sub-block u / (2 MT), row tile, weight tile
                        const int i = u / (2 * MT), m = u / 2 % MT, b = u & 1, ib = 4 * half + i;
                        if constexpr (BLK) {
                            const float d = __fmul_rn(W::d(rec[b]), float(W::scale(rec[b], ib))), off = __fmul_rn(d, -kBias);
                            auto scaled = [&](int q) { return __fmaf_rn(__builtin_bit_cast(float, int(pend[q])), d, off); };
#pragma unroll
                            for (int c = 0; c < 4; ++c) {
                                float * a = &acc[b][m][4 * c];
                                a[0] = __fmaf_rn(scaled(4 * c), pend_s[c].x, a[0]);
                                a[1] = __fmaf_rn(scaled(4 * c + 1), pend_s[c].y, a[1]);
                                a[2] = __fmaf_rn(scaled(4 * c + 2), pend_s[c].z, a[2]);
                                a[3] = __fmaf_rn(scaled(4 * c + 3), pend_s[c].w, a[3]);
                            }
                        } else {
                            const int ls = W::scale(rec[b], ib);
#pragma unroll
                            for (int q = 0; q < 16; ++q) {
                                isum[b][m][q] = (ib == 0 ? 0 : isum[b][m][q]) + __mul24(pend[q], ls);
                                asm("" : "+v"(isum[b][m][q]));   // (sums of several sub-blocks' products would be regrouped, with all of them alive)
                            }
                        }
                    };
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        v4i w[2];
#pragma unroll
                        for (int b = 0; b < 2; ++b) {
                            w[b] = W::operand(code[b][i]);
                            code[b][i] = W::code(c_src[b], st_next * 4 + i, n, g);
                        }
#pragma unroll
                        for (int m = 0; m < MT; ++m) {
                            const v4i a = *reinterpret_cast<const v4i *>(&s_rows[half][m * 4096 + n * 128 + (((2 * i + g) ^ ((n >> 1) & 7)) * 16)]);
                            [[maybe_unused]] float4 sc[4];
                            auto scales = [&](float4 (&to)[4]) {
#pragma unroll
                                for (int c = 0; c < 4; ++c) to[c] = *reinterpret_cast<const float4 *>(&s_bs[half][m * 128 + i * 32 + 8 * c + 4 * g]);
                            };
                            if constexpr (BLK && !kLate) scales(sc);
#pragma unroll
                            for (int b = 0; b < 2; ++b) {
                                const int u = (i * MT + m) * 2 + b;
                                if constexpr (kLate) {
                                    if (u) fold(u - 1);
                                    __builtin_amdgcn_sched_barrier(0);
                                }
                                const v16i p = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, w[b], start, 0, 0, 0);
                                if constexpr (kLate) { if (b == 0) scales(pend_s); }
                                else if (u) fold(u - 1);
                                __builtin_amdgcn_sched_barrier(0);
                                pend = p;
                                if constexpr (BLK && !kLate) {
#pragma unroll
                                    for (int c = 0; c < 4; ++c) pend_s[c] = sc[c];
                                }
                            }
                        }
                    }
                    fold(8 * MT - 1);
                }
                if constexpr (!BLK) {
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const float d = W::d(rec[b]);
#pragma unroll
                        for (int m = 0; m < MT; ++m)
#pragma unroll
                            for (int q = 0; q < 16; ++q) acc[b][m][q] = __fmaf_rn(float(isum[b][m][q]), d, acc[b][m][q]);
                    }
                }
            }
        }
        // Result register 4 c + i of lane (n, g) is input row 8 c + 4 g + i of the row tile, weight row n.
        uint8_t * const tile = s_out[wave];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float scl[16];
#pragma unroll
            for (int c = 0; c < 4; ++c) *reinterpret_cast<float4 *>(&scl[4 * c]) = *reinterpret_cast<const float4 *>(&s_scale[m * 32 + 8 * c + 4 * g]);
            const bool live = wt[0] * 32 < row_lim;   // (zeros past the shared expert's rows)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                uint8_t * to = tile + (8 * (i >> 2) + 4 * g + (i & 3)) * kPitch + n * 2;
                if constexpr (GATEUP) *reinterpret_cast<uint16_t *>(to) = live ? swiglu_half(acc[0][m][i], acc[1][m][i], scl[i], k.glu) : uint16_t(0);
                else {
#pragma unroll
                    for (int b = 0; b < 2; ++b) *reinterpret_cast<uint16_t *>(to + b * 64) = to_half_bits(__fmul_rn(acc[b][m][i], scl[i]));
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if constexpr (GATEUP && BLK) {
                // a row's 32 values are one block: two lanes a row, each the values of sixteen bytes of the operand order
                const int row = lane >> 1, h = lane & 1, asg = s_asg[m * 32 + row];
                float v[16];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const uint4 r = *reinterpret_cast<const uint4 *>(tile + row * kPitch + q * 32 + h * 16);
                    const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        v[q * 8 + 2 * i] = half_bits_to_float(uint16_t(d[i] & 0xFFFFu));
                        v[q * 8 + 2 * i + 1] = half_bits_to_float(uint16_t(d[i] >> 16));
                    }
                }
                float amax = 0.f;
#pragma unroll
                for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
                amax = fmaxf(amax, dpp_f<kDppXor1>(amax));
                const float mul = amax > 0.f ? 127.f / amax : 0.f;
                uint32_t o[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {   // dwords 2 h, 4 + 2 h, 2 h + 1, 5 + 2 h
                    const float * s = v + (q & 1) * 8 + (q >> 1) * 4;
                    o[q] = pack4_q<false>(s[0] * mul, s[1] * mul, s[2] * mul, s[3] * mul);
                }
                if (asg >= 0 && wt[0] < tiles) {
                    *reinterpret_cast<uint4 *>(static_cast<uint8_t *>(k.out) + int64_t(asg) * rows + wt[0] * 32 + h * 16) = make_uint4(o[0], o[1], o[2], o[3]);
                    if (h == 0) k.out_scale[int64_t(asg) * tiles + wt[0]] = amax / 127.f;
                }
            } else {
                constexpr int kLanes = kOutCols / 8, kStep = 64 / kLanes;   // lanes a row, rows a store
#pragma unroll
                for (int q = 0; q < 32 / kStep; ++q) {
                    const int row = q * kStep + lane / kLanes, c = lane % kLanes, asg = s_asg[m * 32 + row];
                    const uint4 w = *reinterpret_cast<const uint4 *>(tile + row * kPitch + c * 16);
                    if (asg >= 0 && (c < 4 ? wt[0] : wt[1]) < tiles) *reinterpret_cast<uint4 *>(static_cast<uint16_t *>(k.out) + int64_t(asg) * rows + wt[0] * 32 + c * 8) = w;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    };
    if (MAX == 1 || cnt <= 32) body(std::integral_constant<int, 1>{});
    else body(std::integral_constant<int, MAX>{});
}

template <uint32_t FMT, bool BLK> void grouped_i8_launch(const GroupedArgs & k, int item_rows, bool gateup, unsigned blocks, hipStream_t s) {
    auto go = [&](auto kernel) { kernel<<<blocks, 256, 0, s>>>(k); };
    if (item_rows == 32) { if (gateup) go(&grouped_i8_k<FMT, BLK, 1, true>); else go(&grouped_i8_k<FMT, BLK, 1, false>); }
    else if (gateup) go(&grouped_i8_k<FMT, BLK, 2, true>);
    else go(&grouped_i8_k<FMT, BLK, 2, false>);
}

}  // namespace
}  // namespace tqmoe
