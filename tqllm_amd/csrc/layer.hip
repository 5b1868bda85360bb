// The whole layer behind one entry point: router -> top-k -> activation image -> gate/up + SwiGLU -> down + combine.
#include <algorithm>

#include "formats.cuh"
#include "grouped_rows_api.cuh"
#include "routing_api.cuh"

namespace tqmoe {
int32_t check_bank(const tqmoe_bank * b, const char * what, tqmoe_error * err);
RowIndex grouped_index(float * scale, int64_t assignments, int experts, int4 ** items);
int32_t enqueue_gather_rows_i8(const int8_t * rq, const float * rs, int cols, const int * counts, const int * offsets, const int * perm, int experts,
                               int64_t assignments, int xdiv, int8_t * q, float * scale, hipStream_t s, float * block_scale, bool indexed);
bool decode_few_takes(const tqmoe_bank & gate, const tqmoe_bank & down, int slots, int shared_ff);
int32_t expert_down_combine(const tqmoe_bank & down, const void * act_image, const int32_t * ids, const float * weights, const float * shared_weights, int32_t n,
                            int32_t slots, int32_t topk, int32_t shared_ff, void * out, uint32_t otype, const void * residual, void * stream, tqmoe_error * err);
bool plane_gemm_has(uint32_t type);
bool plane_gemm_is_fp8(uint32_t type);
// decode.hip: the gate / up products with the clamp of the SwiGLU inputs
int32_t expert_gateup_glu(const tqmoe_bank * gate, const tqmoe_bank * up, const void * x_image, void * act_image, const int32_t * ids, int32_t n,
                          int32_t slots, int32_t topk, int32_t shared_ff, Glu glu, void * stream, tqmoe_error * err, const DecodeTopk & route = DecodeTopk{});
int32_t gemm_8bit_common(const tqmoe_bank * b0, const tqmoe_bank * b1, const int8_t * xq, const float * xs, const int32_t * counts, const int32_t * offsets,
                         const int32_t * perm, int32_t n, int32_t slots, int32_t topk, int32_t shared_lim, void * out, int gateup, void * stream,
                         tqmoe_error * err, const char * what, bool fp8, const float * block_scale, bool blocks, Glu glu, int out_bf16, const float * plan_from);
// the act rows' grouping and the down product read the index that the input rows' grouping built (the same lists)
int32_t group_rows_common(const void * x, uint32_t xtype, int32_t cols, const int32_t * counts, const int32_t * offsets, const int32_t * perm, int32_t experts,
                          int64_t assignments, int32_t xdiv, void * q, float * scale, void * stream, tqmoe_error * err, bool f8, const char * what,
                          float * block_scale, bool blocks, const float * plan_from);
int32_t gemm_f16_common(const tqmoe_bank * b0, const tqmoe_bank * b1, const void * x, uint32_t xtype, const int32_t * counts, const int32_t * offsets,
                        const int32_t * perm, int32_t n, int32_t slots, int32_t topk, int32_t shared_lim, int32_t xdiv, void * out, uint32_t otype, int gateup,
                        void * stream, tqmoe_error * err, const char * what, Glu glu);

namespace {

// From here on the down product of Q4_K banks leaves its rows as halves where the int8 products, which this batch ran on before it
// had products on prepared rows, take the shape (int8_ok) and did the same: the sum over a token's experts reads half the bytes
// (4096 tokens: 45 us of the layer). Everything else keeps fp32 rows: halves end at 65504.
constexpr int kQ4kHalfRows = 2048;
// Where the descriptor asks for the int8 grouped products (act_blocks nonzero), IQ4_XS banks take them from kGroupedMin tokens.
constexpr int kGroupedMin = 64;
// Left to the library (act_blocks zero), IQ4_XS banks take them from kInt8Tokens tokens. The line is where the result changes:
// a scale per token on eight bits moves the layer's result by 2 % of its norm. (4096 tokens of 10 of 512 experts, Zipf / balanced:
// 525 / 611 us a layer with a scale per token, 569 / 620 with the fp16 products on prepared rows; 1500 tokens 315 with a scale per token.)
constexpr int kInt8Tokens = 1024;
// Few tokens: the down blocks add a token's experts themselves, and with plain softmax routing the gate / up blocks select their
// own experts: three launches a layer instead of five (of about 2 us each on the GPU and 3.5 us of host time). An expert that
// several tokens chose is read once for each of them, from the caches, and a block of the down launch walks all of a token's
// weight rows. Where all the down blocks find a compute unit of their own (256 blocks of 32 columns) the three launches are the
// faster ones for every shape (layer in us, five / three, IQ4_XS: 2048 x 768 experts, top-8, two tokens 27.7 / 18.0, four 33.8 /
// 26.2; 4096 x 1024, top-8, two 37.0 / 32.2; 512 x 1024, top-8, twelve 33.1 / 28.0; 7168 x 2048, top-8, one 55.0 / 49.6).
// Beyond, what a launch reads is the line (weights of one projection over all assignments): 2048 x 768, top-8, eight tokens (101 M)
// 44.0 / 36.7, nine (113 M) 45.7 / 47.9; 2048 x 512, top-10 and a shared one, eight (92 M) 49.0 / 38.9, nine (104 M) 49.4 / 49.3; 2048 x
// 1024, top-8, six (101 M) 44.9 / 39.8, seven (117 M) 48.0 / 45.7 (IQ3_S 46.2 / 48.2); 4096 x 1024, top-4, six (101 M) 44.5 / 40.2, seven
// (117 M) 49.3 / 48.2; 3072 x 1024, top-6, six (113 M) 50.1 / 49.7 (Q4_K with Q6_K 46.0 / 52.7); 2048 x 1536, top-6 and a shared one, five
// (110 M) 46.2 / 47.8; 3072 x 1536, top-8 and a shared one, three (127 M) 53.0 / 54.7; 1024 x 512, top-8, twelve (50 M) 32.5 / 28.7. Q6_K's
// gate / up kernel leaves a SIMD two waves: 1024 x 768, top-8 and a shared one, ten tokens 43.5 / 49.2 (2048 x 768, top-8, seven 60.9 / 51.9).
// A token with more than 64 units (super-blocks of its experts' rows) keeps a block's sixteen waves too long (1024 x 4096, top-6, one
// token 28.9 / 36.7).
constexpr int kFewTokens = 12;
bool few_tokens(uint32_t gate_type, int n, int slots, int hidden, int ff) {
    if (n > kFewTokens || slots * (ff / 256) > 64) return false;
    if (int64_t(n) * (hidden / 32) <= 256) return true;           // the down launch's blocks: one a compute unit
    return (gate_type != TQMOE_Q6_K || n <= 7) && int64_t(n) * slots * hidden * ff <= 102000000;
}
constexpr int kDecodeAssignments = 65535;   // per decode launch
constexpr int kDecodeDedup = 2048;          // assignments up to which the decode kernels serve an expert's rows together
constexpr int kGroupedPerBank = 3;          // assignments per expert from which the fp16 grouped products are the faster path

struct Plan {  // byte offsets into the workspace
    bool grouped;   // the grouped products (prefill sizes): int8 for IQ4_XS banks, fp16 for the other formats
    bool int8;
    int chunk;   // tokens per pass of the expert stages
    size_t logits, ids, weights, shared_w, ids_ext, total;
    size_t ximage, aimage, y;                                                // decode path
    size_t xq, xs, counts, offsets, perm, dispatch_ws, act16, aq, as, y16, rq, rs;   // grouped path
    bool blocks;            // int8 products with a scale per 32 activations
    bool few;                // one to a few tokens: the weighted sum inside the down launch
    bool routes;             // ... and the routing inside the gate / up launch
    bool prepared;           // fp16 products on prepared rows
    bool half_rows;          // their down product's rows are halves
    int item_rows;           // rows of their items at most
    size_t x16, xs16, items;
    size_t xbs, abks;        // their block scales
};

bool banks_aligned(const tqmoe_layer & L) { return grouped_rows_aligned(L.gate) && grouped_rows_aligned(L.up) && grouped_rows_aligned(L.down); }
// the 8-bit grouped products: both banks' formats have one with the same operand type (int8, or E4M3 for NVFP4G)
bool int8_ok(const tqmoe_layer & L) {
    return plane_gemm_has(L.gate.type) && plane_gemm_has(L.down.type) && plane_gemm_is_fp8(L.gate.type) == plane_gemm_is_fp8(L.down.type) &&
           (!plane_gemm_is_fp8(L.gate.type) || banks_aligned(L)) && L.hidden % 256 == 0 && L.ff % 256 == 0 && (!L.has_shared || L.shared_ff % 256 == 0);
}

// The descriptor grew three times: one that ends before the routing fields means softmax, normalised, no bias; one that
// ends before act_blocks means a scale per token; one that ends before swiglu_clamp means no clamp.
constexpr size_t kLayerBaseSize = offsetof(tqmoe_layer, gating), kLayerRoutingSize = offsetof(tqmoe_layer, act_blocks);
constexpr size_t kLayerBlocksSize = offsetof(tqmoe_layer, swiglu_clamp);
// the descriptor's request for the int8 grouped products: 0 none (the library chooses), 1 a scale per 32 activations, 2 a scale per token
int int8_mode_of(const tqmoe_layer & L) { return L.struct_size >= kLayerBlocksSize ? (L.act_blocks == 1 ? 1 : L.act_blocks == 2 ? 2 : 0) : 0; }
bool act_blocks_of(const tqmoe_layer & L) { return int8_mode_of(L) == 1; }
// Formats whose 8-bit grouped products are the faster ones at n tokens: the lattice formats of two and three bits that have
// no fp16 products on prepared rows (a tenth faster than the fp16 kernel that takes every format), NVFP4G on its fp8
// products; and IQ4_XS from kInt8Tokens tokens (see there). Q4_K, Q6_K and IQ3_S run on prepared fp16 rows at every size (Q4_K at 4096
// tokens 479 us a layer against 827 on its three int8 planes; IQ3_S at 512 tokens 240 against 391 on its int8
// planes), the others on the general fp16 kernel, 5 to 25 % faster than int8 there.
bool int8_faster(uint32_t type, int n) {
    switch (type) {
        case TQMOE_IQ4_XS: return n >= kInt8Tokens;
        case TQMOE_NVFP4G: case TQMOE_IQ3_XXS: case TQMOE_IQ2_XXS: case TQMOE_IQ2_XS: case TQMOE_IQ2_S: case TQMOE_IQ1_S: return true;
        default: return false;
    }
}
// a descriptor that ends before swiglu_clamp does not clamp
Glu glu_of(const tqmoe_layer & L) { return L.struct_size >= sizeof(tqmoe_layer) ? Glu{L.swiglu_clamp, L.clamp_gate ? 1 : 0} : Glu{0.f, 0}; }

struct Routing { int32_t gating; int32_t norm; const float * bias; };
Routing routing_of(const tqmoe_layer & L) {
    if (L.struct_size < kLayerRoutingSize) return Routing{TQMOE_GATE_SOFTMAX, 1, nullptr};
    return Routing{L.gating ? L.gating : int32_t(TQMOE_GATE_SOFTMAX), L.raw_weights ? 0 : 1, L.probs_bias};
}

Plan plan_for(const tqmoe_layer & L, int n) {
    Plan p{};
    const int slots = L.topk + (L.has_shared ? 1 : 0), banks = L.n_expert + (L.has_shared ? 1 : 0);
    // Few tokens: the decode kernels. From kGroupedPerBank assignments per bank matrix on average the grouped products
    // (measured: the decode kernels' time grows with the assignments, the grouped products' with the experts they decode, and
    // the two cross at about three assignments per expert), and in any case once the decode kernels no longer read every
    // expert's weights once (they group an expert's rows up to kDecodeDedup assignments a launch).
    // Which grouped products: the descriptor's request (act_blocks), else the faster ones for the formats (int8_faster).
    const bool many = int64_t(n) * slots > std::min<int64_t>(kDecodeDedup, int64_t(kGroupedPerBank) * banks);
    const bool iq4xs = L.gate.type == TQMOE_IQ4_XS && L.down.type == TQMOE_IQ4_XS;
    if (int8_mode_of(L) != 0) p.int8 = int8_ok(L) && (iq4xs ? n >= kGroupedMin : many);
    else p.int8 = int8_ok(L) && many && int8_faster(L.gate.type, n) && int8_faster(L.down.type, n);
    p.grouped = p.int8 || many;
    // the grouped products take 2^24 assignments a pass (32-bit block and byte counts stay far from their limits), the
    // decode kernels 65535
    const int64_t per_pass = p.int8 ? int64_t(1) << 24 : p.grouped ? int64_t(65535 - banks) * 64 : kDecodeAssignments;
    p.chunk = int(std::min<int64_t>(n, std::max<int64_t>(1, per_pass / slots)));
    size_t o = 0;
    auto take = [&](size_t bytes) { const size_t at = o; o = align_up(o + bytes, 256); return at; };
    p.logits = take(size_t(n) * (L.n_expert + 1) * 4);
    p.ids = take(size_t(n) * L.topk * 4);
    p.weights = take(size_t(n) * L.topk * 4);
    p.shared_w = take(size_t(n) * 4);
    p.ids_ext = take(size_t(n) * slots * 4);
    const size_t c = size_t(p.chunk), a = c * slots;
    if (p.grouped) {
        p.counts = take(size_t(banks) * 4);
        p.offsets = take(size_t(banks + 1) * 4);
        p.perm = take(a * 4);
        p.dispatch_ws = take(size_t((a + kDispatchChunk - 1) / kDispatchChunk) * banks * sizeof(int));   // the assignments of each chunk's experts
        p.act16 = take(a * L.ff * 2);
        p.y16 = take(a * L.hidden * 4);   // fp16 rows (int8 products) or fp32 rows (fp16 products)
    }
    // the products on prepared rows take both banks: the gate / up product leaves its rows in the order the down product reads
    const bool rows_ok = banks_aligned(L) && grouped_rows_takes(L.gate.type, L.ff, L.hidden) && grouped_rows_takes(L.down.type, L.hidden, L.ff) && (!L.has_shared || L.shared_ff % 128 == 0);
    const bool rows_i8 = banks_aligned(L) && grouped_i8_takes(L.gate.type, L.ff, L.hidden) && grouped_i8_takes(L.down.type, L.hidden, L.ff);
    p.item_rows = grouped_rows_per_item(L.gate.type, int64_t(a), banks);
    if (p.int8 && plane_gemm_is_fp8(L.gate.type)) {
        p.prepared = rows_ok;    // int8_ok's conditions are the stricter ones
        p.rq = take(c * L.hidden);
        p.rs = take(c * 4);
        p.aq = take(a * L.ff);
        p.as = take(a * 4);
        p.items = take(size_t(1 + grouped_rows_items(int64_t(a), banks, p.item_rows)) * sizeof(int4));
    } else if (p.int8 && rows_i8) {
        p.prepared = true;
        p.blocks = act_blocks_of(L);
        p.item_rows = grouped_i8_per_item(p.blocks, int64_t(a), banks);
        p.rq = take(c * L.hidden);
        p.rs = take(c * 4 * (p.blocks ? size_t(L.hidden / 32) : 1));
        p.aq = take(a * L.ff);
        p.as = take(a * 4 * (p.blocks ? size_t(L.ff / 32) : 1));
        p.items = take(size_t(1 + grouped_rows_items(int64_t(a), banks, p.item_rows)) * sizeof(int4));
    } else if (p.int8) {
        const size_t grows = size_t(tqmoe_grouped_rows(int64_t(a), banks));
        p.xq = take(grows * L.hidden);
        const size_t gwords = size_t(tqmoe_grouped_scale_words(int64_t(a), banks));
        p.xs = take(gwords * 4);
        p.aq = take(grows * L.ff);
        p.as = take(gwords * 4);
        p.blocks = act_blocks_of(L);
        p.rq = take(c * L.hidden);        // the chunk's input rows as int8, quantised once, then gathered per assignment
        p.rs = take(c * 4 * (p.blocks ? size_t(L.hidden / 32) : 1));
        if (p.blocks) {
            p.xbs = take(size_t(tqmoe_grouped_block_scale_words(int64_t(a), banks, L.hidden)) * 4);
            p.abks = take(size_t(tqmoe_grouped_block_scale_words(int64_t(a), banks, L.ff)) * 4);
        }
    } else if (p.grouped) {
        p.prepared = rows_ok && !plane_gemm_is_fp8(L.gate.type) && !plane_gemm_is_fp8(L.down.type);
        p.half_rows = L.gate.type == TQMOE_Q4_K && L.down.type == TQMOE_Q4_K && n >= kQ4kHalfRows && int8_ok(L);
        if (p.prepared) {
            p.x16 = take(c * L.hidden * 2);
            p.xs16 = take(c * 4);
            p.items = take(size_t(1 + grouped_rows_items(int64_t(a), banks, p.item_rows)) * sizeof(int4));
        }
    } else {
        const Routing rt = routing_of(L);
        // (rows too wide for the decode products' entry, which refuses them: up to six tokens have the three launches all the same)
        const bool only = n <= 6 && !split_for(L.ff / 32).m;
        p.few = (only || few_tokens(L.gate.type, n, slots, L.hidden, L.ff)) && decode_few_takes(L.gate, L.down, slots, L.has_shared ? L.shared_ff : 0);
        p.routes = p.few && rt.gating == TQMOE_GATE_SOFTMAX && rt.norm && !rt.bias && L.n_expert <= 512 && L.topk <= 64;
        p.ximage = take(tqmoe_act_image_bytes(n, L.hidden));
        p.aimage = take(tqmoe_act_image_bytes(int32_t(a), L.ff));
        p.y = take(a * L.hidden * 4);
    }
    p.total = o;
    return p;
}

int32_t check_layer(const tqmoe_layer * L, tqmoe_error * err) {
    const char * what = "tqmoe_layer_forward";
    if (!L || L->struct_size < kLayerBaseSize) return fail(err, TQMOE_E_ARG, "%s: layer descriptor missing or too small", what);
    const Routing rt = routing_of(*L);
    if (rt.gating < TQMOE_GATE_SOFTMAX || rt.gating > TQMOE_GATE_SQRT_SOFTPLUS) return fail(err, TQMOE_E_UNSUPPORTED, "%s: unsupported gating function %d", what, rt.gating);
    if (L->hidden <= 0 || L->ff <= 0 || L->n_expert <= 0 || L->n_expert > 4096 || L->topk <= 0 || L->topk > L->n_expert || !L->router)
        return fail(err, TQMOE_E_ARG, "%s: invalid layer shape or pointer", what);
    if (L->router_type != TQMOE_F32 && L->router_type != TQMOE_BF16) return fail(err, TQMOE_E_UNSUPPORTED, "%s: router type must be F32 or BF16", what);
    for (const tqmoe_bank * b : {&L->gate, &L->up, &L->down}) if (int32_t rc = check_bank(b, what, err)) return rc;
    const int banks = L->n_expert + (L->has_shared ? 1 : 0);
    if (L->gate.type != L->up.type) return fail(err, TQMOE_E_UNSUPPORTED, "%s: the gate and up banks must share one format (down may have its own)", what);
    if (L->gate.rows != L->ff || L->gate.cols != L->hidden || L->up.rows != L->ff || L->up.cols != L->hidden || L->down.rows != L->hidden ||
        L->down.cols != L->ff || L->gate.experts != banks || L->up.experts != banks || L->down.experts != banks)
        return fail(err, TQMOE_E_ARG, "%s: bank shapes do not match the layer (%d experts of %d x %d expected)", what, banks, L->ff, L->hidden);
    if (L->ff % 32) return fail(err, TQMOE_E_ARG, "%s: ff must be a multiple of 32", what);
    if (L->has_shared && (L->shared_ff <= 0 || L->shared_ff > L->ff || L->shared_ff % 32))
        return fail(err, TQMOE_E_ARG, "%s: shared_ff must be a positive multiple of 32 not above ff", what);
    return 0;
}

}  // namespace
}  // namespace tqmoe

using namespace tqmoe;

extern "C" size_t tqmoe_layer_workspace_bytes(const tqmoe_layer * layer, int32_t n) {
    if (!layer || n <= 0 || check_layer(layer, nullptr)) return 0;
    // Enough for every smaller batch too: a caller asks once, for its largest. A plan's areas grow with the tokens, but at the lines
    // where other products or other items take over their sum may shrink (by up to 29 %: fp16 products in place of the decode
    // products, one expert a token, NVFP4G with a Q6_K down bank).
    const tqmoe_layer & L = *layer;
    const int64_t slots = L.topk + (L.has_shared ? 1 : 0), banks = L.n_expert + (L.has_shared ? 1 : 0);
    size_t most = 0;
    for (int64_t m : {int64_t(n), int64_t(kGroupedMin - 1), int64_t(kInt8Tokens - 1), std::min<int64_t>(kDecodeDedup, kGroupedPerBank * banks) / slots, kItem32 * banks / slots,
                      kItem32Iq3s * banks / slots, kItem64 * banks / slots, kItem32I8 * banks / slots, kItem32I8Blocks * banks / slots})
        if (m > 0 && m <= n) most = std::max(most, plan_for(L, int(m)).total);
    return most + 256;   // (room to move the areas to a multiple of 16 bytes in a workspace that starts elsewhere)
}

extern "C" int32_t tqmoe_layer_path(const tqmoe_layer * layer, int32_t n) {
    if (!layer || n <= 0 || check_layer(layer, nullptr)) return TQMOE_E_ARG;
    const Plan p = plan_for(*layer, n);
    return p.int8 ? (plane_gemm_is_fp8(layer->gate.type) ? TQMOE_PATH_GROUPED_FP8 : TQMOE_PATH_GROUPED_I8) : p.grouped ? TQMOE_PATH_GROUPED_F16 : TQMOE_PATH_DECODE;
}

static int32_t layer_forward(const tqmoe_layer * layer, const void * x, uint32_t xtype, const void * residual, int32_t n, void * out, uint32_t otype,
                             int32_t * ids_out, float * weights_out, float * logits_out, void * workspace, size_t workspace_bytes, void * stream,
                             tqmoe_error * err) {
    if (int32_t rc = check_layer(layer, err)) return rc;
    const tqmoe_layer & L = *layer;
    if (!x || !out || n <= 0) return fail(err, TQMOE_E_ARG, "tqmoe_layer_forward: invalid shape or pointer");
    if (!is_act_type(xtype) || (otype != TQMOE_F32 && otype != TQMOE_BF16)) return fail(err, TQMOE_E_UNSUPPORTED, "tqmoe_layer_forward: unsupported element type");
    const int slots = L.topk + (L.has_shared ? 1 : 0), banks = L.n_expert + (L.has_shared ? 1 : 0);
    const Plan p = plan_for(L, n);
    if (p.grouped && banks > 4096) return fail(err, TQMOE_E_ARG, "tqmoe_layer_forward: the grouped products take at most 4096 experts, the shared one included");   // as tqmoe_dispatch does
    const size_t pad = size_t(-reinterpret_cast<uintptr_t>(workspace)) & 15;
    if (!workspace || workspace_bytes < p.total + pad) return fail(err, TQMOE_E_WORKSPACE, "tqmoe_layer_forward: workspace of %zu bytes needed", p.total + pad);
    if (int32_t rc = need_device(err, "tqmoe_layer_forward")) return rc;
    uint8_t * ws = static_cast<uint8_t *>(workspace) + pad;
    float * logits = logits_out ? logits_out : reinterpret_cast<float *>(ws + p.logits);
    int32_t * ids = ids_out ? ids_out : reinterpret_cast<int32_t *>(ws + p.ids);
    float * weights = weights_out ? weights_out : reinterpret_cast<float *>(ws + p.weights);
    float * shared_w = reinterpret_cast<float *>(ws + p.shared_w);
    const size_t xbytes = elem_bytes(xtype), obytes = elem_bytes(otype);
    const uint8_t * xb = static_cast<const uint8_t *>(x);
    uint8_t * ob = static_cast<uint8_t *>(out);

    if (p.routes) {
        const hipStream_t st = static_cast<hipStream_t>(stream);
        RouterSide side;
        side.image = ws + p.ximage;
        if (int32_t rc = enqueue_router(L.router, L.router_type, L.shared_gate, x, xtype, logits, L.hidden, L.n_expert, n, side, st, err)) return rc;
        const DecodeTopk route{logits, L.n_expert, L.topk, L.has_shared && !L.shared_gate, L.weight_scale, ids, weights, L.has_shared ? shared_w : nullptr};
        if (int32_t rc = expert_gateup_glu(&L.gate, &L.up, ws + p.ximage, ws + p.aimage, nullptr, n, slots, L.topk, L.shared_ff, glu_of(L), stream, err, route)) return rc;
        return expert_down_combine(L.down, ws + p.aimage, ids, weights, shared_w, n, slots, L.topk, L.shared_ff, out, otype, residual, stream, err);
    }
    if (L.hidden % 8) return fail(err, TQMOE_E_ARG, "tqmoe_layer_forward: hidden must be a multiple of 8");
    if ((n + 3) / 4 > 65535) return fail(err, TQMOE_E_ARG, "tqmoe_layer_forward: too many tokens for one call");
    // Beside the routing, in its launches: the rows in the form the products read (a batch that is one pass), the assignments
    // of every dispatch chunk (cleared by the router launch, counted by the top-k launch), the ids extended by the shared expert.
    const hipStream_t hs = static_cast<hipStream_t>(stream);
    const bool whole = p.chunk >= n, counted = p.grouped && whole && banks <= kDispatchWide && L.topk <= 64;
    int * chunk_counts = reinterpret_cast<int *>(ws + p.dispatch_ws);
    RouterSide rside;
    TopkSide side;
    if (counted) {
        rside.zero = side.chunk_counts = chunk_counts;
        rside.zero_n = int((int64_t(n) * slots + kDispatchChunk - 1) / kDispatchChunk) * banks;
        side.banks = banks;
    }
    if (!p.grouped || whole) {
        side.rows = !p.grouped ? kRowsImage : !p.int8 ? (p.prepared ? kRowsHalves : kRowsNone) : plane_gemm_is_fp8(L.gate.type) ? kRowsFp8 : p.blocks ? kRowsInt8Blocks : kRowsInt8;
        side.x = x;
        side.xtype = xtype;
        side.cols = L.hidden;
        side.q = ws + (!p.grouped ? p.ximage : p.int8 ? p.rq : p.x16);
        side.scale = reinterpret_cast<float *>(ws + (p.int8 ? p.rs : p.xs16));
    }
    if (int32_t rc = enqueue_router(L.router, L.router_type, L.shared_gate, x, xtype, logits, L.hidden, L.n_expert, n, rside, hs, err)) return rc;
    int32_t * ext = L.has_shared ? reinterpret_cast<int32_t *>(ws + p.ids_ext) : nullptr;
    const Routing rt = routing_of(L);
    const Glu glu = glu_of(L);
    enqueue_topk(logits, ids, weights, shared_w, ext, L.n_expert, L.n_expert, L.topk, n, L.weight_scale, rt.gating, rt.bias, rt.norm, L.has_shared && !L.shared_gate, side, hs);
    if (int32_t rc = launched(err, "tqmoe_layer_forward (top-k)")) return rc;
    const int32_t * ids_ext = ext ? ext : ids;

    for (int t0 = 0; t0 < n; t0 += p.chunk) {
        const int c = std::min(p.chunk, n - t0);
        const int32_t * cid = ids_ext + size_t(t0) * slots;
        const float * cw = weights + size_t(t0) * L.topk, * csw = shared_w + t0;
        void * cout = ob + size_t(t0) * L.hidden * obytes;
        // the weighted sum of the chunk's rows, with the residual rows added when the caller gave them
        auto combine = [&](const void * routed, uint32_t rtype, const void * shared) -> int32_t {
            if (residual)
                return tqmoe_combine_residual(routed, rtype, slots, shared, int64_t(slots) * L.hidden, cw, csw,
                                              static_cast<const uint8_t *>(residual) + size_t(t0) * L.hidden * 2, cout, L.hidden, L.topk, c, stream, err);
            if (rtype == TQMOE_F16)
                return tqmoe_combine_strided_f16(routed, slots, shared, int64_t(slots) * L.hidden, cw, csw, cout, otype, L.hidden, L.topk, c, stream, err);
            return tqmoe_combine_strided(static_cast<const float *>(routed), slots, static_cast<const float *>(shared), int64_t(slots) * L.hidden, cw, csw, cout, otype,
                                         L.hidden, L.topk, c, stream, err);
        };
        if (p.grouped) {
            int8_t * xq = reinterpret_cast<int8_t *>(ws + p.xq), * aq = reinterpret_cast<int8_t *>(ws + p.aq);
            float * xs = reinterpret_cast<float *>(ws + p.xs), * as = reinterpret_cast<float *>(ws + p.as);
            int32_t * counts = reinterpret_cast<int32_t *>(ws + p.counts), * offsets = reinterpret_cast<int32_t *>(ws + p.offsets),
                    * perm = reinterpret_cast<int32_t *>(ws + p.perm);
            uint16_t * act16 = reinterpret_cast<uint16_t *>(ws + p.act16), * y16 = reinterpret_cast<uint16_t *>(ws + p.y16);
            DispatchSide lists;
            lists.counted = counted;
            if (p.prepared) {
                lists.item_rows = p.item_rows;
                lists.items = reinterpret_cast<int4 *>(ws + p.items);
            } else if (p.int8) {
                lists.item_rows = 128;
                lists.index = grouped_index(xs, int64_t(c) * slots, banks, &lists.items);
            }
            if (int32_t rc = enqueue_layer_dispatch(cid, counts, offsets, perm, banks, c, slots, chunk_counts, lists, hs, err)) return rc;
            if (p.prepared && p.int8) {   // 8-bit rows: E4M3 or int8
                uint8_t * rq = ws + p.rq, * aq = ws + p.aq;
                float * rs = reinterpret_cast<float *>(ws + p.rs), * as = reinterpret_cast<float *>(ws + p.as);
                int4 * items = reinterpret_cast<int4 *>(ws + p.items);
                const int shared_expert = L.has_shared ? banks - 1 : -1;
                const int64_t a = int64_t(c) * slots;
                const void * xc = xb + size_t(t0) * L.hidden * xbytes;
                const Glu none{0.f, 0};
                if (plane_gemm_is_fp8(L.gate.type)) {
                    if (!whole)
                        if (int32_t rc = tqmoe_quant_rows_fp8(xc, xtype, c, L.hidden, rq, rs, stream, err)) return rc;
                    enqueue_grouped_products(L.gate, &L.up, rq, rs, perm, items, a, slots, act16, false, shared_expert, L.shared_ff, glu, hs, p.item_rows);
                    if (int32_t rc = tqmoe_quant_rows_fp8(act16, TQMOE_F16, a, L.ff, aq, as, stream, err)) return rc;
                    enqueue_grouped_products(L.down, nullptr, aq, as, perm, items, a, 1, y16, false, shared_expert, L.shared_ff, none, hs, p.item_rows);
                } else {
                    int8_t * rq8 = reinterpret_cast<int8_t *>(rq), * aq8 = reinterpret_cast<int8_t *>(aq);
                    if (!whole) {
                        const int32_t rc = p.blocks ? tqmoe_quant_rows_i8_blocks(xc, xtype, c, L.hidden, rq8, rs, nullptr, stream, err) : tqmoe_quant_rows_i8(xc, xtype, c, L.hidden, rq8, rs, stream, err);
                        if (rc) return rc;
                    }
                    if (p.blocks) {   // (a weight tile's act values are one block: the gate / up product quantises them)
                        enqueue_grouped_i8(L.gate, &L.up, rq8, rs, true, perm, items, a, slots, aq8, as, shared_expert, L.shared_ff, glu, hs, p.item_rows);
                    } else {
                        enqueue_grouped_i8(L.gate, &L.up, rq8, rs, false, perm, items, a, slots, act16, nullptr, shared_expert, L.shared_ff, glu, hs, p.item_rows);
                        if (int32_t rc = tqmoe_quant_rows_i8(act16, TQMOE_F16, a, L.ff, aq8, as, stream, err)) return rc;
                    }
                    enqueue_grouped_i8(L.down, nullptr, aq8, as, p.blocks, perm, items, a, 1, y16, nullptr, shared_expert, L.shared_ff, none, hs, p.item_rows);
                }
                if (int32_t rc = launched(err, "tqmoe_layer_forward (grouped products)")) return rc;
                if (int32_t rc = combine(y16, TQMOE_F16, L.has_shared ? y16 + size_t(L.topk) * L.hidden : nullptr)) return rc;
                continue;
            }
            if (p.prepared) {
                const hipStream_t st = static_cast<hipStream_t>(stream);
                uint16_t * x16 = reinterpret_cast<uint16_t *>(ws + p.x16);
                float * xs16 = reinterpret_cast<float *>(ws + p.xs16);
                int4 * items = reinterpret_cast<int4 *>(ws + p.items);
                const int shared_expert = L.has_shared ? banks - 1 : -1;
                const int64_t a = int64_t(c) * slots;
                if (!whole) enqueue_prepare_rows(xb + size_t(t0) * L.hidden * xbytes, xtype, c, L.hidden, x16, xs16, st);
                enqueue_grouped_products(L.gate, &L.up, x16, xs16, perm, items, a, slots, act16, false, shared_expert, L.shared_ff, glu, st, p.item_rows);
                enqueue_grouped_products(L.down, nullptr, act16, nullptr, perm, items, a, 1, y16, !p.half_rows, shared_expert, L.shared_ff, Glu{0.f, 0}, st, p.item_rows);
                if (int32_t rc = launched(err, "tqmoe_layer_forward (grouped products)")) return rc;
                const uint8_t * yb = ws + p.y16;
                if (int32_t rc = combine(yb, p.half_rows ? TQMOE_F16 : TQMOE_F32, L.has_shared ? yb + size_t(L.topk) * L.hidden * (p.half_rows ? 2 : 4) : nullptr)) return rc;
                continue;
            }
            if (!p.int8) {
                if (int32_t rc = gemm_f16_common(&L.gate, &L.up, xb + size_t(t0) * L.hidden * xbytes, xtype, counts, offsets, perm, c, slots, L.topk, L.shared_ff, slots,
                                                 act16, TQMOE_F16, 1, stream, err, "tqmoe_layer_forward (gate / up)", glu)) return rc;
                float * y32 = reinterpret_cast<float *>(y16);
                if (int32_t rc = tqmoe_expert_gemm(&L.down, act16, TQMOE_F16, counts, offsets, perm, c, slots, L.topk, L.shared_ff, 1, y32, TQMOE_F32, stream, err)) return rc;
                if (int32_t rc = combine(y32, TQMOE_F32, L.has_shared ? y32 + size_t(L.topk) * L.hidden : nullptr)) return rc;
                continue;
            } else {
            int8_t * rq = reinterpret_cast<int8_t *>(ws + p.rq);
            float * rs = reinterpret_cast<float *>(ws + p.rs);
            if (p.blocks) {
            float * xbs = reinterpret_cast<float *>(ws + p.xbs), * abks = reinterpret_cast<float *>(ws + p.abks);
            if (!whole)
                if (int32_t rc = tqmoe_quant_rows_i8_blocks(xb + size_t(t0) * L.hidden * xbytes, xtype, c, L.hidden, rq, rs, nullptr, stream, err)) return rc;
            enqueue_gather_rows_i8(rq, rs, L.hidden, counts, offsets, perm, banks, int64_t(c) * slots, slots, xq, xs, hs, xbs, true);
            if (int32_t rc = gemm_8bit_common(&L.gate, &L.up, xq, xs, counts, offsets, perm, c, slots, L.topk, L.shared_ff, act16, 1, stream, err,
                                              "tqmoe_layer_forward (gate / up)", false, xbs, true, glu, 0, nullptr)) return rc;
            if (int32_t rc = group_rows_common(act16, TQMOE_F16, L.ff, counts, offsets, perm, banks, int64_t(c) * slots, 1, aq, as, stream, err, false,
                                               "tqmoe_layer_forward (act rows)", abks, true, xs)) return rc;
            if (int32_t rc = gemm_8bit_common(&L.down, nullptr, aq, as, counts, offsets, perm, c, slots, L.topk, L.shared_ff, y16, 0, stream, err,
                                              "tqmoe_layer_forward (down)", false, abks, true, Glu{0.f, 0}, 0, xs)) return rc;
            } else {
            if (!whole)
                if (int32_t rc = tqmoe_quant_rows_i8(xb + size_t(t0) * L.hidden * xbytes, xtype, c, L.hidden, rq, rs, stream, err)) return rc;
            enqueue_gather_rows_i8(rq, rs, L.hidden, counts, offsets, perm, banks, int64_t(c) * slots, slots, xq, xs, hs, nullptr, true);
            if (int32_t rc = gemm_8bit_common(&L.gate, &L.up, xq, xs, counts, offsets, perm, c, slots, L.topk, L.shared_ff, act16, 1, stream, err,
                                              "tqmoe_layer_forward (gate / up)", false, nullptr, false, glu, 0, nullptr)) return rc;
            if (int32_t rc = group_rows_common(act16, TQMOE_F16, L.ff, counts, offsets, perm, banks, int64_t(c) * slots, 1, aq, as, stream, err, false,
                                               "tqmoe_layer_forward (act rows)", nullptr, false, xs)) return rc;
            if (int32_t rc = gemm_8bit_common(&L.down, nullptr, aq, as, counts, offsets, perm, c, slots, L.topk, L.shared_ff, y16, 0, stream, err,
                                              "tqmoe_layer_forward (down)", false, nullptr, false, Glu{0.f, 0}, 0, xs)) return rc;
            }
            }
            if (int32_t rc = combine(y16, TQMOE_F16, L.has_shared ? y16 + size_t(L.topk) * L.hidden : nullptr)) return rc;
        } else {
            const uint8_t * ximage = ws + p.ximage + tqmoe_act_image_bytes(1, L.hidden) * size_t(t0);
            float * y = reinterpret_cast<float *>(ws + p.y);
            if (int32_t rc = expert_gateup_glu(&L.gate, &L.up, ximage, ws + p.aimage, cid, c, slots, L.topk, L.shared_ff, glu, stream, err)) return rc;
            if (p.few) return expert_down_combine(L.down, ws + p.aimage, ids, weights, shared_w, n, slots, L.topk, L.shared_ff, out, otype, residual, stream, err);
            if (int32_t rc = tqmoe_expert_down(&L.down, ws + p.aimage, y, cid, c, slots, L.topk, L.shared_ff, stream, err)) return rc;
            if (int32_t rc = combine(y, TQMOE_F32, L.has_shared ? y + size_t(L.topk) * L.hidden : nullptr)) return rc;
        }
    }
    return ok(err);
}

extern "C" int32_t tqmoe_layer_forward(const tqmoe_layer * layer, const void * x, uint32_t xtype, int32_t n, void * out, uint32_t otype,
                                       int32_t * ids_out, float * weights_out, float * logits_out, void * workspace, size_t workspace_bytes,
                                       void * stream, tqmoe_error * err) {
    return layer_forward(layer, x, xtype, nullptr, n, out, otype, ids_out, weights_out, logits_out, workspace, workspace_bytes, stream, err);
}

extern "C" int32_t tqmoe_layer_forward_residual(const tqmoe_layer * layer, const void * x, uint32_t xtype, const void * residual, int32_t n, void * out,
                                                int32_t * ids_out, float * weights_out, float * logits_out, void * workspace, size_t workspace_bytes,
                                                void * stream, tqmoe_error * err) {
    if (!residual) return fail(err, TQMOE_E_ARG, "tqmoe_layer_forward_residual: residual rows missing");
    return layer_forward(layer, x, xtype, residual, n, out, TQMOE_BF16, ids_out, weights_out, logits_out, workspace, workspace_bytes, stream, err);
}
