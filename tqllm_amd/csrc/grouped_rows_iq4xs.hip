// The grouped fp16 products on prepared rows of IQ4_XS banks.
#include "grouped_rows_kernels.cuh"

namespace tqmoe {
template <uint32_t FMT> void grouped_rows_run(const GroupedArgs & k, int item_rows, bool gateup, bool f32_out, unsigned blocks, hipStream_t s);
template <> void grouped_rows_run<TQMOE_IQ4_XS>(const GroupedArgs & k, int item_rows, bool gateup, bool f32_out, unsigned blocks, hipStream_t s) {
    grouped_rows_launch<TQMOE_IQ4_XS>(k, item_rows, gateup, f32_out, blocks, s);
}
}  // namespace tqmoe
