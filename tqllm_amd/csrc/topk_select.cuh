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
// first `rounds` selections. x: the token's logits; lane l owns entries l, l + 64, ...
// Every round is a chain of dependent wave reductions, so the rounds carry only what the next round needs: the winner's key
// stays in lane s and the probabilities are computed for all selections at once afterwards. Equal keys are rare: one ballot
// tells whether the winner is alone, and only a tie pays for the index reduction.
template <int R> __device__ __forceinline__ void topk_select(const float * __restrict__ x, int e, int rounds, int lane, bool weights, int & my_id, float & my_w) {
    int key[R];
    float m = -INFINITY, sum = 0.f;
    {
        float l[R];
#pragma unroll
        for (int r = 0; r < R; ++r) { const int j = lane + 64 * r; l[r] = j < e ? x[j] : -INFINITY; m = fmaxf(m, l[r]); }
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
