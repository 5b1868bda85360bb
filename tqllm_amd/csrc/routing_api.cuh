// What the layer asks of the routing launches beside the routing (routing.hip): work on the same rows or ids that would
// otherwise be launches of their own.
#pragma once
#include "grouped_rows_api.cuh"

namespace tqmoe {

constexpr int kDispatchChunk = 1024;        // consecutive assignments a dispatch block places
constexpr int kDispatchWide = 1024;         // experts up to which it does so in one launch
constexpr int kRouterFew = 7;               // tokens up to which the router takes them one a pass

struct RouterSide {
    uint8_t * image = nullptr;              // activation images of the rows (batches of one-token passes only)
    int * zero = nullptr;                   // ints to clear: the per-chunk counts the top-k launch adds to
    int zero_n = 0;
};
enum { kRowsNone = 0, kRowsImage, kRowsHalves, kRowsFp8, kRowsInt8, kRowsInt8Blocks };
struct TopkSide {
    int rows = kRowsNone;                   // form the input rows are written in
    const void * x = nullptr;
    uint32_t xtype = 0;
    int cols = 0;
    void * q = nullptr;                     // the rows
    float * scale = nullptr;                // their scales
    int * chunk_counts = nullptr;           // [chunks][banks], cleared before: += 1 per assignment
    int banks = 0;
};
// behind the lists: the grouped products' items and the gathered rows' index
struct DispatchSide {
    bool counted = false;                   // chunk_counts hold the counts already
    int item_rows = 0;                      // 0: no plan
    int4 * items = nullptr;
    RowIndex index{};
};

int32_t enqueue_router(const void * router, uint32_t wtype, const void * shared_gate, const void * x, uint32_t xtype, float * logits, int hidden, int experts, int n,
                       const RouterSide & side, hipStream_t s, tqmoe_error * err);
int32_t enqueue_topk(const float * logits, int32_t * ids, float * weights, float * shared_weights, int32_t * ext_ids, int32_t extra, int32_t experts, int32_t topk, int32_t n,
                     float scale, int32_t gating, const float * bias, int32_t norm, int32_t shared_ungated, const TopkSide & side, hipStream_t s);
int32_t enqueue_layer_dispatch(const int32_t * ids, int32_t * counts, int32_t * offsets, int32_t * perm, int32_t experts, int32_t n, int32_t topk, int * chunk_counts,
                               const DispatchSide & side, hipStream_t s, tqmoe_error * err);

}  // namespace tqmoe
