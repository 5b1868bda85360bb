// Grouped products on prepared rows: row preparation, the plan of items, the launches (kernels: grouped_rows_kernels.cuh).
#include "grouped_rows_api.cuh"
#include "formats.cuh"
#include "grouped_plan.cuh"
#include "row_quant.cuh"

namespace tqmoe {
namespace {

template <int XT>
__global__ __launch_bounds__(256) void prepare_rows_k(const void * __restrict__ x, int64_t rows, int cols, uint16_t * __restrict__ out, float * __restrict__ xs) {
    const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row < rows) prepare_row_wave<XT>(x, row, cols, out, xs, threadIdx.x & 63);
}

__global__ __launch_bounds__(1024) void grouped_plan_k(const int * __restrict__ counts, const int * __restrict__ offsets, int experts, int item_rows, int4 * __restrict__ plan, RowIndex index) {
    plan_items(counts, offsets, experts, item_rows, plan, index);
}

}  // namespace

template <uint32_t FMT> void grouped_rows_run(const GroupedArgs & k, int item_rows, bool gateup, bool f32_out, unsigned blocks, hipStream_t s);

// Rows of an item at most. 128 spread a weight's decode over four row tiles; 64 need 168 registers in place of 256, three waves
// a SIMD in place of two, which is what counts where most experts have a row tile or two. fp16 products, layer in us at 64 /
// 128 rows, balanced and Zipf routing: IQ3_S, 256 experts with 16 rows 210 / 234 and 160 / 177, with 35 rows 273 / 297 and 238 / 243,
// with 40 rows 282 / 304 and 262 / 258; IQ4_XS, 77 experts with 40 rows 196 / 203 and 203 / 206, 128 with 35 rows 165 / 175 and 161 / 155, with
// 40 rows 178 / 181 and 169 / 168; Q6_K, 77 with 40 rows 210 / 214 and 231 / 224; Q4_K, 64 experts with 44 rows 98 / 102 and 109 / 126, with 60
// rows 119 / 116 and 124 / 140; Q4_K / Q6_K, 128 experts with 42 rows 177 / 183 and 182 / 177, with 84 rows 264 / 248 and 261 / 242.
// 32, of the formats whose items of one row tile keep the super-block's factor out of the operands: all items have one then, in three
// waves a SIMD, but an expert's weights are decoded for every 32 of its rows, which Zipf routing's popular experts feel. At 32 / 64 rows:
// IQ4_XS, 512 experts with 3 rows 247 / 281 and 87 / 95, with 7 rows 272 / 295 and 126 / 126 (128 rows, Zipf: 116, which the averages cannot
// tell), with 14 rows 283 / 301 and 171 / 168, with 22 rows 298 / 321 and 240 / 221, 128 experts with 22 rows 139 / 150 and 129 / 130, with 30 rows
// 147 / 161 and 159 / 157, with 35 rows 167 / 165 and 175 / 161, 77 experts with 30 rows 181 / 177 and 179 / 174; Q6_K, 77 experts with 10 rows
// 171 / 172 and 126 / 151, with 22 rows 195 / 188 and 171 / 181, with 30 rows 200 / 198 and 205 / 199. IQ3_S (64 rows: whole weights, three waves), 256
// experts with 8 rows 199 / 203 and 115 / 121, with 16 rows 206 / 210 and 172 / 160, with 22 rows 231 / 231 and 218 / 188.
// The fp8 products' codes leave LDS for two blocks either way: 128.
int grouped_rows_per_item(uint32_t type, int64_t assignments, int experts) {
    const int one_tile = type == TQMOE_IQ4_XS || type == TQMOE_Q6_K ? kItem32 : type == TQMOE_IQ3_S ? kItem32Iq3s : 0;
    if (assignments <= int64_t(experts) * one_tile) return 32;
    return type != TQMOE_NVFP4G && assignments <= int64_t(experts) * kItem64 ? 64 : 128;
}

bool grouped_rows_takes(uint32_t type, int rows, int cols) {
    return (type == TQMOE_IQ4_XS || type == TQMOE_Q4_K || type == TQMOE_Q6_K || type == TQMOE_IQ3_S || type == TQMOE_NVFP4G) && rows % 32 == 0 && cols % 256 == 0;
}

void enqueue_prepare_rows(const void * x, uint32_t xtype, int64_t rows, int cols, uint16_t * out, float * xs, hipStream_t s) {
    const unsigned blocks = unsigned((rows + 3) / 4);
    switch (xtype) {
        case TQMOE_F32: prepare_rows_k<TQMOE_F32><<<blocks, 256, 0, s>>>(x, rows, cols, out, xs); break;
        case TQMOE_F16: prepare_rows_k<TQMOE_F16><<<blocks, 256, 0, s>>>(x, rows, cols, out, xs); break;
        default: prepare_rows_k<TQMOE_BF16><<<blocks, 256, 0, s>>>(x, rows, cols, out, xs); break;
    }
}

void enqueue_grouped_plan(const int * counts, const int * offsets, int experts, int item_rows, int4 * plan, const RowIndex & index, hipStream_t s) {
    grouped_plan_k<<<1, 1024, 0, s>>>(counts, offsets, experts, item_rows, plan, index);
}

// assignments: total entries of perm (it bounds the items)
void enqueue_grouped_products(const tqmoe_bank & b0, const tqmoe_bank * b1, const void * x, const float * xs, const int * perm, const int4 * plan, int64_t assignments,
                         int xdiv, void * out, bool f32_out, int shared_expert, int shared_lim, Glu glu, hipStream_t s, int item_rows, bool row_tiles) {
    const int tiles = b0.rows / 32, per = b1 ? 4 : 8, groups = (tiles + per - 1) / per;
    const GroupedArgs k{view(b0), b1 ? view(*b1) : view(b0), x, xs, perm, plan, xdiv, out, groups, shared_expert, shared_lim, glu, row_tiles, nullptr};
    // (an XCD takes an eighth of every one of the four classes, rounded up)
    const unsigned blocks = unsigned((grouped_rows_items(assignments, b0.experts, item_rows) + 28) / 8 * 8 * groups);
    switch (b0.type) {
        case TQMOE_IQ4_XS: grouped_rows_run<TQMOE_IQ4_XS>(k, item_rows, b1 != nullptr, f32_out, blocks, s); break;
        case TQMOE_Q4_K: grouped_rows_run<TQMOE_Q4_K>(k, item_rows, b1 != nullptr, f32_out, blocks, s); break;
        case TQMOE_Q6_K: grouped_rows_run<TQMOE_Q6_K>(k, item_rows, b1 != nullptr, f32_out, blocks, s); break;
        case TQMOE_NVFP4G: grouped_rows_run<TQMOE_NVFP4G>(k, item_rows, b1 != nullptr, f32_out, blocks, s); break;
        default: grouped_rows_run<TQMOE_IQ3_S>(k, item_rows, b1 != nullptr, f32_out, blocks, s); break;
    }
}

}  // namespace tqmoe
