// The grouped fp16 products on prepared rows of Q4_K banks.
#include "grouped_f16_kernels.cuh"

namespace tqmoe {
template <uint32_t FMT> void grouped_f16_run(const GroupedF16Args & k, bool gateup, bool f32_out, unsigned blocks, hipStream_t s);
template <> void grouped_f16_run<TQMOE_Q4_K>(const GroupedF16Args & k, bool gateup, bool f32_out, unsigned blocks, hipStream_t s) {
    grouped_f16_launch<TQMOE_Q4_K>(k, gateup, f32_out, blocks, s);
}
}  // namespace tqmoe
