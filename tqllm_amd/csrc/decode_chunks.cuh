// The input rows a decode block serves: assignments that share an expert are cut into chunks, so that a chunk's block
// reads (and decodes) the expert's weights once for all of the chunk's rows.
#pragma once
#include "common.cuh"

namespace tqmoe {

constexpr int kChunkRowsMax = 4;   // input rows per block at most

// The block's own expert, e = ids[a], and the assignments it serves. mode 0: its own only. mode 1: the assignments of ids[0..A) with its
// expert, in index order, are cut into chunks of kChunkRowsMax; the block of each chunk's first assignment serves the chunk (returns its
// size and the assignment indices in tok, -1 past the end) and the other blocks leave (returns 0, as for an id that is negative).
// Every wave finds this by itself, in scalar registers: 512 ids in one trip to memory, a ballot for 64 of them. (One wave that walks a
// copy of the ids in LDS, for the others to read behind two barriers, took 5000 cycles of a block's 30000 with 176 assignments, 7800 of
// 54000 with 512.)
__device__ __forceinline__ int chunk_rows(const int * __restrict__ ids, int A, int a, int mode, int & e, int (&tok)[kChunkRowsMax]) {
    e = ids[a];
#pragma unroll
    for (int j = 0; j < kChunkRowsMax; ++j) tok[j] = -1;
    if (mode == 0) { tok[0] = a; return e < 0 ? 0 : 1; }
    const int lane = threadIdx.x & 63;
    int rank = 0, n = 0;
    for (int i0 = 0; i0 < A && n < kChunkRowsMax; i0 += 512) {
        int v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = ids[min(i0 + q * 64 + lane, A - 1)];
        if (e < 0) return 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int base = i0 + q * 64;
            if (base >= A) break;
            unsigned long long mask = __ballot(v[q] == e && base + lane < A);
            if (base + 64 <= a) { rank += __popcll(mask); continue; }
            if (base <= a) {
                const unsigned long long before = (1ull << (a - base)) - 1ull;
                rank += __popcll(mask & before);
                if (rank % kChunkRowsMax) return 0;
                mask &= ~before;
            }
#pragma unroll
            for (int j = 0; j < kChunkRowsMax; ++j)
                if (n == j && mask) { tok[j] = base + __ffsll(mask) - 1; mask &= mask - 1ull; ++n; }
        }
    }
    return n;
}

}  // namespace tqmoe
