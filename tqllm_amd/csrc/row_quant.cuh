// Input rows in the forms the grouped products read, a wave a row: 8-bit with a scale, or fp16 in operand order.
#pragma once
#include "act_image.cuh"
#include "grouped_rows_api.cuh"

namespace tqmoe {
namespace {

// four scaled values -> four operand bytes: int8 (round to nearest) or E4M3 (round to nearest even; the values are
// clamped to +-448 first, so the conversion never leaves the finite codes)
template <bool F8> __device__ __forceinline__ uint32_t pack4_q(float a, float b, float c, float d) {
    if constexpr (F8) {
        auto clamp = [](float v) { return fminf(fmaxf(v, -448.f), 448.f); };
        int w = __builtin_amdgcn_cvt_pk_fp8_f32(clamp(a), clamp(b), 0, false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(clamp(c), clamp(d), w, true);
        return uint32_t(w);
    } else {
        return uint32_t(__float2int_rn(a) & 0xFF) | uint32_t(__float2int_rn(b) & 0xFF) << 8 | uint32_t(__float2int_rn(c) & 0xFF) << 16 |
               uint32_t(__float2int_rn(d) & 0xFF) << 24;
    }
}
template <bool F8> constexpr float kOperandMax = F8 ? 448.f : 127.f;

// the largest magnitude over the four lanes that hold a 32-value block (eight values each)
__device__ __forceinline__ float quad_max(float v) {
    v = fmaxf(v, dpp_f<kDppXor1>(v));
    return fmaxf(v, dpp_f<kDppXor2>(v));
}
__device__ __forceinline__ int byte_sum_i8(uint32_t w) { return int(int8_t(w)) + int(int8_t(w >> 8)) + int(int8_t(w >> 16)) + int(int8_t(w >> 24)); }

// A row's pieces of eight values that a lane takes (lane, lane + 64, ...): the first kRowKeep are loaded together and stay in registers,
// so a row of up to 3072 values is one trip to memory; a longer one's rest is read again where it is needed.
// Without KEEP both passes read memory: less code, and code that runs once is fetched from memory too, so a lane's int8 conversions, three
// times an E4M3 code's instructions, are not laid out six times. us a launch, read twice / kept: 8192 rows of 3072 bf16 beside the
// selection to E4M3 23.0 / 20.2, 65536 of 1536 fp16 to E4M3 64.3 / 53.5, 4096 of 2048 fp32 beside the selection to fp16 14.3 / 13.0; to
// int8 4096 of 2048 bf16 beside the selection 12.6 / 13.2, 45056 of 512 fp16 16.8 / 17.2.
constexpr int kRowKeep = 6;
template <int XT, bool KEEP> struct RowPieces {
    static constexpr int kKept = KEEP ? kRowKeep : 0, kOwn = KEEP ? kRowKeep : 1;
    static constexpr int kRaw = XT == TQMOE_F32 ? 2 : 1, kSize = XT == TQMOE_F32 ? 4 : 2;
    uint4 raw[kOwn][kRaw];
    const uint8_t * row;
    int pieces, lane;
    __device__ __forceinline__ RowPieces(const void * x, int64_t r, int cols, int l) : row(static_cast<const uint8_t *>(x) + r * cols * kSize), pieces(cols / 8), lane(l) {
#pragma unroll
        for (int p = 0; p < kKept; ++p) {
            if (64 * p >= pieces) break;
            const int at = min(64 * p + lane, pieces - 1);
#pragma unroll
            for (int h = 0; h < kRaw; ++h) raw[p][h] = *reinterpret_cast<const uint4 *>(row + (int64_t(at) * kRaw + h) * 16);
        }
    }
    // f(piece, its values) for every piece of the lane
    template <typename F> __device__ __forceinline__ void each(const F & f) const {
#pragma unroll
        for (int p = 0; p < kKept; ++p) {
            if (64 * p >= pieces) return;
            const int at = 64 * p + lane;
            float v[8];
            load8<XT>(raw[p], 0, v);
            if (at < pieces) f(at, v);
        }
        for (int at = 64 * kKept + lane; at < pieces; at += 64) {
            float v[8];
            load8<XT>(row, int64_t(at) * 8, v);
            f(at, v);
        }
    }
    __device__ __forceinline__ float lane_max() const {
        float amax = 0.f;
        each([&](int, const float (&v)[8]) {
#pragma unroll
            for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
        });
        return amax;
    }
};

// One wave: a row of 8-bit activations: q = rint(x * 127 / amax) per row, scale = amax / 127 (E4M3: 448 in place of 127).
// BLK: amax and scale per block of 32 values (scale [rows][cols / 32]) and, when asked for, the sums of q over each 16
// values (qsum [rows][cols / 32][2]).
template <int XT, bool F8, bool BLK>
__device__ __forceinline__ void quant_row_wave(const void * __restrict__ x, int64_t row, int cols, int8_t * __restrict__ q, float * __restrict__ scale,
                                               int16_t * __restrict__ qsum, int lane) {
    if constexpr (BLK) {           // (a block's four lanes enter or leave the loop together: cols is a multiple of 32)
        const int groups = cols / 8;   // 8 consecutive values = natural dwords 2j, 2j + 1 of a 32-block
        uint32_t * out = reinterpret_cast<uint32_t *>(q + row * cols);
        for (int gi = lane; gi < groups; gi += 64) {
            float v[8];
            load8<XT>(x, row * cols + gi * 8, v);
            float amax = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
            amax = quad_max(amax);
            const float mul = amax > 0.f ? 127.f / amax : 0.f;
            const uint32_t w[2] = {pack4_q<false>(v[0] * mul, v[1] * mul, v[2] * mul, v[3] * mul), pack4_q<false>(v[4] * mul, v[5] * mul, v[6] * mul, v[7] * mul)};
            const int blk = gi >> 2, d0 = 2 * (gi & 3);
            out[blk * 8 + plane_pos(d0)] = w[0];
            out[blk * 8 + plane_pos(d0 + 1)] = w[1];
            if ((gi & 3) == 0) scale[row * (cols / 32) + blk] = amax / 127.f;
            if (qsum) {
                int sum = byte_sum_i8(w[0]) + byte_sum_i8(w[1]);
                sum += dpp_i<kDppXor1>(sum);
                if ((gi & 1) == 0) qsum[(row * (cols / 32) + blk) * 2 + ((gi & 3) >> 1)] = int16_t(sum);
            }
        }
        return;
    }
    const RowPieces<XT, F8> in(x, row, cols, lane);
    float amax = in.lane_max();
    amax = fmaxf(amax, dpp_f<kDppXor1>(amax));
    amax = fmaxf(amax, dpp_f<kDppXor2>(amax));
    amax = fmaxf(amax, dpp_f<kDppHalfMirror>(amax));
    amax = fmaxf(amax, dpp_f<kDppMirror>(amax));
    amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
    const float mul = amax > 0.f ? kOperandMax<F8> / amax : 0.f;
    if (lane == 0) scale[row] = amax / kOperandMax<F8>;
    uint32_t * out = reinterpret_cast<uint32_t *>(q + row * cols);
    in.each([&](int gi, const float (&v)[8]) {
        const uint32_t w[2] = {pack4_q<F8>(v[0] * mul, v[1] * mul, v[2] * mul, v[3] * mul), pack4_q<F8>(v[4] * mul, v[5] * mul, v[6] * mul, v[7] * mul)};
        const int blk = gi >> 2, d0 = 2 * (gi & 3);
        out[blk * 8 + plane_pos(d0)] = w[0];
        out[blk * 8 + plane_pos(d0 + 1)] = w[1];
    });
}

// One wave: an input row -> fp16 in operand order (operand_pos). A row whose largest magnitude leaves the middle of
// fp16's range is scaled by a power of two (exact), which the product's epilogue takes back: xs[row].
template <int XT>
__device__ __forceinline__ void prepare_row_wave(const void * __restrict__ x, int64_t row, int cols, uint16_t * __restrict__ out, float * __restrict__ xs, int lane) {
    const RowPieces<XT, true> in(x, row, cols, lane);
    const float amax = wave_max(in.lane_max());
    float back = 1.f, mul = 1.f;
    if (amax > 16384.f || (amax < 0.0078125f && amax > 0.f)) {
        int ex;
        (void)frexpf(amax, &ex);
        ex = max(min(ex, 126), -126);
        back = ldexpf(1.f, ex);
        mul = ldexpf(1.f, -ex);
    }
    if (lane == 0) xs[row] = back;
    uint2 * o = reinterpret_cast<uint2 *>(out + row * cols);
    in.each([&](int p, const float (&v)[8]) {
        auto two = [&](float a, float b) { return uint32_t(__half_as_ushort(__float2half_rn(a * mul))) | uint32_t(__half_as_ushort(__float2half_rn(b * mul))) << 16; };
        // values 8 q .. 8 q + 7 of block p / 4: dwords j = 2 (q % 2) and j + 1, halves q / 2
        const int q = p & 3, j = 2 * (q & 1), h = q >> 1;
        uint2 * b = o + (p >> 2) * 8;
        b[2 * j + h] = make_uint2(two(v[0], v[2]), two(v[1], v[3]));
        b[2 * (j + 1) + h] = make_uint2(two(v[4], v[6]), two(v[5], v[7]));
    });
}

}  // namespace
}  // namespace tqmoe
