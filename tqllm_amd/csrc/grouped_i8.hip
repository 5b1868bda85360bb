// The grouped int8 products on rows in quantiser order (kernels: grouped_i8_kernels.cuh).
#include "grouped_i8_kernels.cuh"

namespace tqmoe {

bool grouped_i8_takes(uint32_t type, int rows, int cols) { return type == TQMOE_IQ4_XS && rows % 32 == 0 && cols % 256 == 0; }

// Rows of an item at most: 64 decode a weight once for two row tiles, 32 need 168 registers in place of 242, three waves a SIMD in
// place of two, which is the better where most experts have one row tile. Layer in us at 32 / 64 rows, a scale per 32 values: 512
// experts with 22 rows on average 272 / 291, 32 rows 337 / 337, 36 rows 377 / 368 (Zipf 310 / 295), 41 rows 414 / 395, 64 rows 522 / 498;
// 128 experts with 36 rows 151 / 158, 42 rows 170 / 169; a scale a row: 22 rows 261 / 276, 32 rows 323 / 319, 43 rows 438 / 386.
int grouped_i8_per_item(bool blocks, int64_t assignments, int experts) { return assignments <= int64_t(experts) * (blocks ? kItem32I8Blocks : kItem32I8) ? 32 : 64; }

// assignments: total entries of perm (it bounds the items)
void enqueue_grouped_i8(const tqmoe_bank & b0, const tqmoe_bank * b1, const int8_t * x, const float * xs, bool blocks, const int * perm, const int4 * plan, int64_t assignments,
                        int xdiv, void * out, float * out_scale, int shared_expert, int shared_lim, Glu glu, hipStream_t s, int item_rows) {
    const int tiles = b0.rows / 32, per = b1 ? 4 : 8, groups = (tiles + per - 1) / per;
    const GroupedArgs k{view(b0), b1 ? view(*b1) : view(b0), x, xs, perm, plan, xdiv, out, groups, shared_expert, shared_lim, glu, 0, out_scale};
    // (an XCD takes an eighth of every one of the four classes, rounded up)
    const unsigned grid = unsigned((grouped_rows_items(assignments, b0.experts, item_rows) + 28) / 8 * 8 * groups);
    if (blocks) grouped_i8_launch<TQMOE_IQ4_XS, true>(k, item_rows, b1 != nullptr, grid, s);
    else grouped_i8_launch<TQMOE_IQ4_XS, false>(k, item_rows, b1 != nullptr, grid, s);
}

}  // namespace tqmoe
