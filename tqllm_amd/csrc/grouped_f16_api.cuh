// Types shared by the grouped fp16 products on prepared rows: the entry (grouped_f16.hip) and the per-format kernels.
#pragma once
#include "decode_api.cuh"

namespace tqmoe {

constexpr int kGroupedRows = 128;   // input rows of an item at most

// Where value i of 32 lies in a prepared row: eight halves (one operand read) are the values the matrix operand of code dword
// j holds, 4 j .. 4 j + 3 and 16 + 4 j .. 16 + 4 j + 3, each four in the order 0, 2, 1, 3 (the pairs that one mask or
// byte permute takes out of a dword of codes).
__host__ __device__ constexpr int operand_pos(int i) { return ((i >> 2) & 3) * 8 + (i >> 4) * 4 + ((i & 1) << 1) + ((i >> 1) & 1); }

struct GroupedF16Args {
    BankView b0, b1;          // gate and up; down: the same bank twice
    const uint16_t * x;       // prepared rows, cols halves each
    const float * xs;         // their scales, or null (all 1)
    const int * perm;         // assignment indices grouped by expert
    const int4 * plan;        // entry 0: number of items; then per item: expert, first index into perm, rows
    int xdiv;                 // row of assignment a = a / xdiv
    void * out;               // gate / up: prepared rows [assignments][rows] for the down product; else rows of fp32 or halves
    int groups;               // blocks per item: groups of weight tiles
    int shared_expert;        // the expert whose rows (gate / up) or columns (down) stop at shared_lim, or -1
    int shared_lim;
    Glu glu;
};

bool grouped_f16_takes(uint32_t type, int rows, int cols);
inline int64_t grouped_f16_items(int64_t assignments, int experts) { return assignments / kGroupedRows + experts; }   // at most

}  // namespace tqmoe
