// Grouped products on prepared rows: row preparation, the plan of items, the launches (kernels: grouped_rows_kernels.cuh).
#include "grouped_rows_api.cuh"
#include "formats.cuh"

namespace tqmoe {
namespace {

// Input rows -> fp16 rows in operand order (operand_pos), a wave a row. A row whose largest magnitude leaves the middle of
// fp16's range is scaled by a power of two (exact), which the product's epilogue takes back: xs[row].
template <int XT>
__global__ __launch_bounds__(256) void prepare_rows_k(const void * __restrict__ x, int64_t rows, int cols, uint16_t * __restrict__ out, float * __restrict__ xs) {
    const int lane = threadIdx.x & 63;
    const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int pieces = cols / 8;
    float amax = 0.f;
    for (int p = lane; p < pieces; p += 64) {
        float v[8];
        load8<XT>(x, row * cols + p * 8, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    }
    amax = wave_max(amax);
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
    for (int p = lane; p < pieces; p += 64) {
        float v[8];
        load8<XT>(x, row * cols + p * 8, v);
        auto two = [&](float a, float b) { return uint32_t(__half_as_ushort(__float2half_rn(a * mul))) | uint32_t(__half_as_ushort(__float2half_rn(b * mul))) << 16; };
        // values 8 q .. 8 q + 7 of block p / 4: dwords j = 2 (q % 2) and j + 1, halves q / 2
        const int q = p & 3, j = 2 * (q & 1), h = q >> 1;
        uint2 * b = o + (p >> 2) * 8;
        b[2 * j + h] = make_uint2(two(v[0], v[2]), two(v[1], v[3]));
        b[2 * (j + 1) + h] = make_uint2(two(v[4], v[6]), two(v[5], v[7]));
    }
}

// Items of the products: an expert's rows cut into runs of item_rows, the full runs of all experts first, then the rests by
// row tiles (four and three, two, one): the last blocks of a launch are its short ones. Where index is given, the index of
// the gathered row tiles (RowIndex) too.
constexpr int kScans = 6;   // full runs, rests of three classes; row tiles, chunks of chunk_tiles of them
__global__ __launch_bounds__(1024) void grouped_plan_k(const int * __restrict__ counts, const int * __restrict__ offsets, int experts, int item_rows, int4 * __restrict__ plan, RowIndex index) {
    __shared__ int s_wave[kScans][16];
    __shared__ int s_total[kScans];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (experts + 1023) / 1024, lo = min(tid * per, experts), hi = min(lo + per, experts);
    auto rest_class = [](int rest) { return rest > 64 ? 1 : rest > 32 ? 2 : rest > 0 ? 3 : -1; };
    auto add = [&](int c, int (&v)[kScans]) {
        const int k = rest_class(c % item_rows), t = (c + 31) / 32;
        v[0] += c / item_rows;
#pragma unroll
        for (int i = 1; i < 4; ++i) v[i] += k == i;
        v[4] += t;
        if (index.tile_base) v[5] += (t + index.chunk_tiles - 1) / index.chunk_tiles;
    };
    int mine[kScans] = {};
    for (int e = lo; e < hi; ++e) add(max(counts[e], 0), mine);
    int at[kScans];
#pragma unroll
    for (int i = 0; i < kScans; ++i) {
        int v = mine[i];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) { const int u = __shfl_up(v, d, 64); if (lane >= d) v += u; }
        at[i] = v - mine[i];
        if (lane == 63) s_wave[i][wave] = v;
    }
    __syncthreads();
    if (tid < kScans) {
        int sum = 0;
        for (int w = 0; w < 16; ++w) { const int v = s_wave[tid][w]; s_wave[tid][w] = sum; sum += v; }
        s_total[tid] = sum;
    }
    __syncthreads();
    int base = 0;
#pragma unroll
    for (int i = 0; i < kScans; ++i) { at[i] += s_wave[i][wave] + (i < 4 ? base : 0); if (i < 4) base += s_total[i]; }
    if (tid == 0) {
        plan[0] = make_int4(s_total[0], s_total[1], s_total[2], s_total[3]);
        if (index.tile_base) { index.tile_base[experts] = s_total[4]; index.chunk_base[experts] = s_total[5]; }
    }
    if (index.tile_base && tid < index.counters_n) index.counters[tid] = 0;
    for (int e = lo; e < hi; ++e) {
        const int c = max(counts[e], 0), first = offsets[e], full = c / item_rows, rest = c % item_rows;
        for (int f = 0; f < full; ++f) plan[1 + at[0] + f] = make_int4(e, first + f * item_rows, item_rows, at[4] + f * (item_rows / 32));
        const int k = rest_class(rest);
#pragma unroll
        for (int i = 1; i < 4; ++i) if (k == i) plan[1 + at[i]] = make_int4(e, first + full * item_rows, rest, at[4] + full * (item_rows / 32));
        if (index.tile_base) { index.tile_base[e] = at[4]; index.chunk_base[e] = at[5]; }
        add(c, at);
    }
}

}  // namespace

template <uint32_t FMT> void grouped_rows_run(const GroupedArgs & k, int item_rows, bool gateup, bool f32_out, unsigned blocks, hipStream_t s);

// Rows of an item at most. 128 spread a weight's decode over four row tiles; 64 need 168 registers in place of 256, three waves
// a SIMD in place of two, which is what counts where most experts have a row tile or two. fp16 products, layer in us at 64 /
// 128 rows: 16 rows an expert (IQ3_S, 512 tokens) 245 / 266, 27 rows 376 / 395, 32 rows 108 / 110, 64 rows 143 / 137; 7 rows
// an expert on average but Zipf routing (IQ4_XS, 333 tokens) 161 / 152, which the averages cannot tell. (32 rows and four
// waves: 238, 382, 121, 160 and 173.) The fp8 products' codes leave LDS for two blocks either way: 128.
int grouped_rows_per_item(uint32_t type, int64_t assignments, int experts) {
    return type != TQMOE_NVFP4G && assignments <= int64_t(experts) * 32 ? 64 : 128;
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
                         int xdiv, void * out, bool f32_out, int shared_expert, int shared_lim, Glu glu, hipStream_t s, int item_rows, bool row_tiles, bool out_bf16) {
    const int tiles = b0.rows / 32, per = b1 ? 4 : 8, groups = (tiles + per - 1) / per;
    const GroupedArgs k{view(b0), b1 ? view(*b1) : view(b0), x, xs, perm, plan, xdiv, out, groups, shared_expert, shared_lim, glu, row_tiles, out_bf16};
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
