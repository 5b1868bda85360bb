// Selection of a token's top-k experts by one wave, shared by the top-k kernels and the decode products that route by themselves.
#pragma once
#include "common.cuh"

namespace tqmoe {
namespace {

template <int CTRL, int ROWS> __device__ __forceinline__ float dpp_keep_f(float v) {   // lanes outside ROWS get their own value back
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, ROWS, 0xF, false));
}
template <int CTRL, int ROWS> __device__ __forceinline__ int dpp_keep_i(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xF, false); }
__device__ __forceinline__ float wave_max_all(float v) {   // the wave's maximum, the same in every lane
    v = fmaxf(v, dpp_f<kDppXor1>(v));
    v = fmaxf(v, dpp_f<kDppXor2>(v));
    v = fmaxf(v, dpp_f<kDppHalfMirror>(v));
    v = fmaxf(v, dpp_f<kDppMirror>(v));
    v = fmaxf(v, dpp_keep_f<0x142, 0xA>(v));   // row_bcast:15 into rows 1 and 3
    v = fmaxf(v, dpp_keep_f<0x143, 0xC>(v));   // row_bcast:31 into rows 2 and 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ int wave_min_all(int v) {
    v = min(v, dpp_i<kDppXor1>(v));
    v = min(v, dpp_i<kDppXor2>(v));
    v = min(v, dpp_i<kDppHalfMirror>(v));
    v = min(v, dpp_i<kDppMirror>(v));
    v = min(v, dpp_keep_i<0x142, 0xA>(v));
    v = min(v, dpp_keep_i<0x143, 0xC>(v));
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max_all_i(int v) {
    v = max(v, dpp_i<kDppXor1>(v));
    v = max(v, dpp_i<kDppXor2>(v));
    v = max(v, dpp_i<kDppHalfMirror>(v));
    v = max(v, dpp_i<kDppMirror>(v));
    v = max(v, dpp_keep_i<0x142, 0xA>(v));
    v = max(v, dpp_keep_i<0x143, 0xC>(v));
    return __builtin_amdgcn_readlane(v, 63);
}
// Selection keys of the softmax top-k. The reference orders by rounded probability, ties to the lower index
// (src/experts/moe.cpp:73-78); exp and the division by the common sum are monotone, so ordering by logit gives the same
// choice whatever exp() the device has, except where two different logits round to one probability. Entries whose
// probability underflowed to zero are all tied there and go by index: they share one key below every logit's.
// A finite float maps to an integer with the same order (-0 counts as +0); the map is its own inverse.
constexpr int kKeyGone = INT_MIN, kKeyZero = INT_MIN + 1;
__device__ __forceinline__ int order_key(float x) { const int i = __float_as_int(x + 0.f); return i ^ ((i >> 31) & 0x7FFFFFFF); }
__device__ __forceinline__ float key_value(int k) { return __int_as_float(k ^ ((k >> 31) & 0x7FFFFFFF)); }

__device__ __forceinline__ float wave_sum_all(float v) {
    v = row_sum16(v);
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xA, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x143, 0xC, 0xF, false));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// One wave, k <= 64 and e <= 64 R: lane s gets selection s (its expert, its softmax probability where `weights` asks for it) for the
// first `rounds` selections. cand: 256 ints in LDS of the wave's own, 16 bytes aligned.
// A wave reduction for the maximum of every selection is a chain of 60 dependent instructions each with eight entries a lane (10 of 512:
// 4900 cycles). So, beyond 128 entries: the `rounds`-th largest of the lanes' maxima is a bound that no selection lies below, and
// few other entries lie above it. A search over the keys, eight parts a step, finds a bound that six maxima more reach at most;
// what reaches it goes to a lane each and counts the larger ones (3000 cycles, more than half of them the fetch of instructions
// that run once: the layer of one token 17.5 -> 17.2 us, 333 tokens 128.8 -> 126.6). Up to 128 entries the rounds are short: eight of 64 take
// 2260 cycles, and the layer of one token 15.9 us with them against 16.4. Where two of what reaches the bound are equal, a
// round for every selection.
template <int R> struct TopkLogits { float l[R]; };   // lane l's entries l, l + 64, ... (-infinity past the end)
template <int R> __device__ __forceinline__ TopkLogits<R> topk_logits(const float * __restrict__ x, int e, int lane) {
    TopkLogits<R> v;
#pragma unroll
    for (int r = 0; r < R; ++r) { const int j = lane + 64 * r; v.l[r] = j < e ? x[j] : -INFINITY; }
    return v;
}
template <int R> __device__ __forceinline__ void topk_select(const TopkLogits<R> & x, int e, int rounds, int lane, bool weights, int * cand, int & my_id, float & my_w) {
    int key[R];
    float m = -INFINITY, sum = 0.f;
    {
        const float (&l)[R] = x.l;
#pragma unroll
        for (int r = 0; r < R; ++r) m = fmaxf(m, l[r]);
        m = wave_max_all(m);
        // (the order alone needs the exponentials only where one may be zero, or a logit is not finite)
        bool far = false;
#pragma unroll
        for (int r = 0; r < R; ++r) far |= lane + 64 * r < e && !(l[r] - m >= -80.f);
        if (weights || __any(far)) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int j = lane + 64 * r;
                const float ex = j < e ? expf(l[r] - m) : 0.f;
                sum += ex;
                key[r] = j < e ? (ex > 0.f ? order_key(l[r]) : kKeyZero) : kKeyGone;   // entries past the end never win
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) key[r] = lane + 64 * r < e ? order_key(l[r]) : kKeyGone;
        }
    }
    int my_key = kKeyZero;
    my_id = 0;
    bool alone = false;
    if constexpr (R > 2) {
        int most = key[0];
#pragma unroll
        for (int r = 1; r < R; ++r) most = max(most, key[r]);
        int low = wave_min_all(most), high = order_key(m) + 1, reach = 64;   // `rounds` maxima or more reach low, fewer high
        for (int i = 0; i < 4 && reach > rounds + 6; ++i) {
            const uint32_t step = (uint32_t(high) - uint32_t(low)) >> 3;
            if (step == 0) break;
            unsigned long long mask[7];
#pragma unroll
            for (int q = 0; q < 7; ++q) mask[q] = __ballot(most >= int(uint32_t(low) + (q + 1) * step));
            __builtin_amdgcn_sched_barrier(0);             // (seven comparisons, then seven counts: a chain each would be waited for in turn)
            int parts = 0;
#pragma unroll
            for (int q = 0; q < 7; ++q) {
                const int c = __popcll(mask[q]);
                if (c >= rounds) { reach = c; parts = q + 1; }
            }
            low = int(uint32_t(low) + parts * step);
            if (parts < 7) high = int(uint32_t(low) + step);
        }
        int total = 0;
        cand[lane] = kKeyGone;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool in = key[r] >= low;
            const unsigned long long mask = __ballot(in);
            const int to = __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), total));
            int * slot = cand + (in && to < 64 ? to : 64 + lane);
            slot[0] = key[r];
            slot[128] = lane + 64 * r + 1;
            total += __popcll(mask);
        }
        alone = total <= 64;
        if (alone) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int own = cand[lane], id1 = cand[128 + lane];
            int before = 0;                            // larger keys; all of them for a lane without an entry
            for (int c = 0; c < total; c += 8) {
                const int4 u = *reinterpret_cast<const int4 *>(cand + c), v = *reinterpret_cast<const int4 *>(cand + c + 4);
                before += (u.x > own) + (u.y > own) + (u.z > own) + (u.w > own) + (v.x > own) + (v.y > own) + (v.z > own) + (v.w > own);
            }
            my_key = __builtin_amdgcn_ds_permute(before * 4, own);
            my_id = __builtin_amdgcn_ds_permute(before * 4, id1) - 1;
            // (two equal keys leave the place behind them empty)
            alone = !__any(lane <= rounds && lane < total && my_id < 0);
        }
    }
    if (!alone) {                                  // equal keys: a round for every selection
        for (int s = 0; s < rounds; ++s) {
            int bk = key[0], bi = lane;
#pragma unroll
            for (int r = 1; r < R; ++r) if (key[r] > bk) { bk = key[r]; bi = lane + 64 * r; }   // strict: the lowest index of equal keys
            const int topkey = wave_max_all_i(bk);
            const unsigned long long tie = __ballot(bk == topkey);
            const int best = __popcll(tie) == 1 ? __builtin_amdgcn_readlane(bi, __builtin_ctzll(tie)) : wave_min_all(bk == topkey ? bi : 0x7FFFFFFF);
            if (lane == s) { my_id = best; my_key = topkey; }
#pragma unroll
            for (int r = 0; r < R; ++r) if (lane + 64 * r == best) key[r] = kKeyGone;
        }
    }
    my_w = 0.f;
    if (weights) {
        sum = wave_sum_all(sum);
        my_w = my_key == kKeyZero ? 0.f : expf(key_value(my_key) - m) / sum;   // the probability, as every entry's would be computed
    }
}
// lane s's share of the selected weights, in slot order as the host sums them, times the scale
__device__ __forceinline__ float topk_weight(float my_w, int k, float scale) {
    float selected = 0.f;
    for (int s = 0; s < k; ++s) selected += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_w), s));
    float v = my_w / fmaxf(selected, 6.103515625e-5f);   // the host divides by the clamped sum, then multiplies by the scale
    if (scale != 0.f && scale != 1.f) v *= scale;
    return v;
}

}  // namespace
}  // namespace tqmoe
