// The grouped fp16 products on prepared rows of Q4_K banks.
#include "grouped_rows_kernels.cuh"

namespace tqmoe {
template <uint32_t FMT> void grouped_rows_run(const GroupedArgs & k, int item_rows, bool gateup, bool f32_out, unsigned blocks, hipStream_t s);
template <> void grouped_rows_run<TQMOE_Q4_K>(const GroupedArgs & k, int item_rows, bool gateup, bool f32_out, unsigned blocks, hipStream_t s) {
    grouped_rows_launch<TQMOE_Q4_K>(k, item_rows, gateup, f32_out, blocks, s);
}
}  // namespace tqmoe
