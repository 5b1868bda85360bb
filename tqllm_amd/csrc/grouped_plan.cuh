// The items of the grouped products from the experts' counts, by one block of 1024 threads.
#pragma once
#include "grouped_rows_api.cuh"

namespace tqmoe {
namespace {

// Items of the products: an expert's rows cut into runs of item_rows, the full runs of all experts first, then the rests by
// row tiles (four and three, two, one): the last blocks of a launch are its short ones. But the rest of an expert with a few full
// runs comes right behind them: its weights, which may be more than an L2 holds, are then read from memory once and not again
// near the launch's end (NVFP4G, 8192 tokens, about 288 rows an expert: 3.3 GB fetched a gate / up launch of 1.45 GB of weights, layer
// 1797 -> 1698 us; Q4_K, 4096 tokens 479 -> 469). With all rests there, or with many full runs in front, the launch ends on long
// items (IQ4_XS, 4096 tokens, Zipf: 526 -> 541). Where index is given, the index of the gathered row tiles (RowIndex) too.
constexpr int kManyItems = 8;
constexpr int kScans = 6;   // full runs, rests of three classes; row tiles, chunks of chunk_tiles of them
__device__ __forceinline__ void plan_items(const int * __restrict__ counts, const int * __restrict__ offsets, int experts, int item_rows, int4 * __restrict__ plan, RowIndex index) {
    __shared__ int s_wave[kScans][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per = (experts + 1023) / 1024, lo = min(tid * per, experts), hi = min(lo + per, experts);
    const int shift = 31 - __clz(item_rows);   // (a power of two)
    auto rest_class = [&](int c) {
        const int full = c >> shift, rest = c & (item_rows - 1);
        return rest == 0 ? -1 : full >= 1 && full < kManyItems ? 0 : rest > 64 ? 1 : rest > 32 ? 2 : 3;
    };
    auto add = [&](int c, int (&v)[kScans]) {
        const int k = rest_class(c), t = (c + 31) / 32;
        v[0] += c >> shift;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += k == i;
        v[4] += t;
        if (index.tile_base) v[5] += (t + index.chunk_tiles - 1) / index.chunk_tiles;
    };
    int mine[kScans] = {};
    for (int e = lo; e < hi; ++e) add(max(counts[e], 0), mine);
    int at[kScans];
#pragma unroll
    for (int i = 0; i < kScans; ++i) {
        const int v = wave_scan(mine[i]);
        at[i] = v - mine[i];
        if (lane == 63) s_wave[i][wave] = v;
    }
    __syncthreads();
    // every wave adds the sixteen waves' sums of all scans by itself: four scans in the rows of one register, two in another's
    const int first = row_scan(s_wave[lane >> 4][lane & 15]), second = row_scan(s_wave[4 + ((lane >> 4) & 1)][lane & 15]);
    int before[kScans], total[kScans];
#pragma unroll
    for (int i = 0; i < kScans; ++i) {
        const int from = i < 4 ? first : second, row = 16 * (i & 3);
        before[i] = wave ? __builtin_amdgcn_readlane(from, row + wave - 1) : 0;
        total[i] = __builtin_amdgcn_readlane(from, row + 15);
    }
    int base = 0;
#pragma unroll
    for (int i = 0; i < kScans; ++i) { at[i] += before[i] + (i < 4 ? base : 0); if (i < 4) base += total[i]; }
    if (tid == 0) {
        plan[0] = make_int4(total[0], total[1], total[2], total[3]);
        if (index.tile_base) { index.tile_base[experts] = total[4]; index.chunk_base[experts] = total[5]; }
    }
    if (index.tile_base && tid < index.counters_n) index.counters[tid] = 0;
    for (int e = lo; e < hi; ++e) {
        const int c = max(counts[e], 0), first = offsets[e], full = c >> shift, rest = c & (item_rows - 1);
        for (int f = 0; f < full; ++f) plan[1 + at[0] + f] = make_int4(e, first + f * item_rows, item_rows, at[4] + f * (item_rows / 32));
        const int k = rest_class(c);
#pragma unroll
        for (int i = 0; i < 4; ++i) if (k == i) plan[1 + at[i] + (i ? 0 : full)] = make_int4(e, first + full * item_rows, rest, at[4] + full * (item_rows / 32));
        if (index.tile_base) { index.tile_base[e] = at[4]; index.chunk_base[e] = at[5]; }
        add(c, at);
    }
}

}  // namespace
}  // namespace tqmoe
