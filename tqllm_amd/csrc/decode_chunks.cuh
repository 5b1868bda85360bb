// The input rows a decode block serves: assignments that share an expert are cut into chunks, so that a chunk's block
// reads (and decodes) the expert's weights once for all of the chunk's rows.
#pragma once
#include "common.cuh"

namespace tqmoe {

constexpr int kChunkRowsMax = 4;   // input rows per block at most

// the first x lanes of a wave
__device__ __forceinline__ unsigned long long first_lanes(int x) { return x <= 0 ? 0ull : ~0ull >> (64 - min(x, 64)); }

// The block's own expert, e = ids[a], and the assignments it serves. mode 0: its own only. mode 1: the assignments of ids[0..A) with its
// expert, in index order, are cut into chunks of kChunkRowsMax; the block of each chunk's first assignment serves the chunk (returns its
// size and the assignment indices in tok, -1 past the end) and the other blocks leave (returns 0, as for an id that is negative).
// Every wave finds this by itself, in scalar registers: up to 192 or 512 ids and its own expert in one trip to memory, a ballot for 64 of
// them, a closer look only at groups that hold the expert. (The expert by a scalar load is waited for before the ids' loads go out, a second
// trip; returns inside the search, and the code of eight groups in the way of the few that a short batch needs, make most of the rest. us, one wave
// that walks a copy of the ids in LDS / every wave, in that form / so: IQ4_XS, 512 experts, down 1024 x 256, 12 tokens of 8 10.3 / 10.7 / 10.2,
// 32 of 8 17.5 / 18.3 / 17.3, 139 of 10 39.2 / 41.8 / 35.5; 2048 x 512, 5 of 4 10.1 / 10.25 / 9.9, 139 of 10 87.9 / 88.4 / 79.4, gate and up 132 / 130 /
// 122. 1 to 139 tokens, ten shapes, five formats: level with the walk in that form, 3.6 % faster so.)
__device__ __forceinline__ int chunk_rows(const int * __restrict__ ids, int A, int a, int mode, int & e, int (&tok)[kChunkRowsMax]) {
#pragma unroll
    for (int j = 0; j < kChunkRowsMax; ++j) tok[j] = -1;
    if (mode == 0) {
        e = ids[a];
        tok[0] = a;
        return e < 0 ? 0 : 1;
    }
    const int lane = threadIdx.x & 63;
    int at = a, rank = 0, n = 0;
    asm volatile("" : "+v"(at));       // (a scalar load would be waited for before the others go out)
    const int own = ids[at];
    auto look = [&](auto groups, int i0) {   // at ids[i0 .. i0 + 64 * groups)
        constexpr int G = decltype(groups)::value;
        int v[G];
#pragma unroll
        for (int q = 0; q < G; ++q) {
            v[q] = -1;
            if (i0 + q * 64 < A) v[q] = ids[min(i0 + q * 64 + lane, A - 1)];
        }
        e = __builtin_amdgcn_readfirstlane(own);
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const int base = i0 + q * 64;
            const unsigned long long same = base < A ? __ballot(v[q] == e) : 0ull;
            if (same) {
                const unsigned long long all = same & first_lanes(A - base), before = first_lanes(a - base);
                rank += __popcll(all & before);
                unsigned long long rest = all & ~before;
#pragma unroll 1
                while (rest && n < kChunkRowsMax) {
                    const int t = base + __ffsll(rest) - 1;
#pragma unroll
                    for (int j = 0; j < kChunkRowsMax; ++j) tok[j] = n == j ? t : tok[j];
                    rest &= rest - 1ull;
                    ++n;
                }
            }
        }
    };
    if (A <= 192) look(std::integral_constant<int, 3>{}, 0);
    else
#pragma unroll 1
        for (int i0 = 0;; i0 += 512) {
            look(std::integral_constant<int, 8>{}, i0);
            if (i0 + 512 >= A || n == kChunkRowsMax || e < 0 || (i0 + 512 > a && rank % kChunkRowsMax)) break;
        }
    return e < 0 || rank % kChunkRowsMax ? 0 : n;
}

}  // namespace tqmoe
