// Types shared by the grouped products on prepared rows: the entry (grouped_rows.hip) and the per-format kernels.
#pragma once
#include "decode_api.cuh"

namespace tqmoe {

// Where value i of 32 lies in a prepared row: eight halves (one operand read) are the values the matrix operand of code dword
// j holds, 4 j .. 4 j + 3 and 16 + 4 j .. 16 + 4 j + 3, each four in the order 0, 2, 1, 3 (the pairs that one mask or
// byte permute takes out of a dword of codes).
__host__ __device__ constexpr int operand_pos(int i) { return ((i >> 2) & 3) * 8 + (i >> 4) * 4 + ((i & 1) << 1) + ((i >> 1) & 1); }

struct GroupedArgs {
    BankView b0, b1;          // gate and up; down: the same bank twice
    const void * x;           // prepared rows: cols halves in operand_pos order, or (NVFP4G) cols E4M3 bytes in the order tqmoe_quant_rows_fp8 leaves
    const float * xs;         // their scales, or null (all 1)
    const int * perm;         // assignment indices grouped by expert
    const int4 * plan;        // entry 0: items of each class (grouped_plan_k); then per item: expert, first index into perm, rows, first row tile
    int xdiv;                 // row of assignment a = a / xdiv
    void * out;               // gate / up: rows of halves [assignments][rows], in operand_pos order (NVFP4G: in natural order); else rows of fp32 or halves
    int groups;               // blocks per item: groups of weight tiles
    int shared_expert;        // the expert whose rows (gate / up) or columns (down) stop at shared_lim, or -1
    int shared_lim;
    Glu glu;
    int row_tiles;            // NVFP4G: x is in operand-major row tiles (each expert's rows padded to whole tiles), xs by row of those
    float * out_scale;        // int8 gate / up with a scale per 32 values: the scales of the act rows, [assignments][rows / 32]
};

// index of the gathered row tiles, written beside the items where tile_base is not null
struct RowIndex { int * tile_base, * chunk_base, * counters; int counters_n, chunk_tiles; };

// Rows an expert on average up to which items are of 32 rows (IQ4_XS and Q6_K; IQ3_S), of 64 (grouped_rows_per_item); int8 ones of 32, with a
// scale a row and per 32 values (grouped_i8_per_item)
constexpr int kItem32 = 24, kItem32Iq3s = 16, kItem64 = 40, kItem32I8 = 28, kItem32I8Blocks = 36;

bool grouped_rows_takes(uint32_t type, int rows, int cols);
inline bool grouped_rows_aligned(const tqmoe_bank & b) { return aligned16(b.codes) && aligned16(b.aux); }   // planes that lie otherwise have the general products
int grouped_rows_per_item(uint32_t type, int64_t assignments, int experts);   // input rows of an item at most: 32, 64 or 128 (type: the gate bank's)
inline int64_t grouped_rows_items(int64_t assignments, int experts, int item_rows) { return assignments / item_rows + experts; }   // at most

void enqueue_prepare_rows(const void * x, uint32_t xtype, int64_t rows, int cols, uint16_t * out, float * xs, hipStream_t s);
void enqueue_grouped_plan(const int * counts, const int * offsets, int experts, int item_rows, int4 * plan, const RowIndex & index, hipStream_t s);
// assignments: total entries of perm (it bounds the items)
void enqueue_grouped_products(const tqmoe_bank & b0, const tqmoe_bank * b1, const void * x, const float * xs, const int * perm, const int4 * plan, int64_t assignments,
                              int xdiv, void * out, bool f32_out, int shared_expert, int shared_lim, Glu glu, hipStream_t s, int item_rows, bool row_tiles = false);

// int8 products on rows in quantiser order (a row per token or per assignment); blocks: a scale per 32 values
bool grouped_i8_takes(uint32_t type, int rows, int cols);
int grouped_i8_per_item(bool blocks, int64_t assignments, int experts);   // input rows of an item at most: 32 or 64
void enqueue_grouped_i8(const tqmoe_bank & b0, const tqmoe_bank * b1, const int8_t * x, const float * xs, bool blocks, const int * perm, const int4 * plan, int64_t assignments,
                        int xdiv, void * out, float * out_scale, int shared_expert, int shared_lim, Glu glu, hipStream_t s, int item_rows);

}  // namespace tqmoe
