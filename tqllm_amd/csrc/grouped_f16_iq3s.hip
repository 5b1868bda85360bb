// The grouped fp16 products on prepared rows of IQ3_S banks.
#include "grouped_f16_kernels.cuh"

namespace tqmoe {
template <uint32_t FMT> void grouped_f16_run(const GroupedF16Args & k, bool gateup, bool f32_out, unsigned blocks, hipStream_t s);
template <> void grouped_f16_run<TQMOE_IQ3_S>(const GroupedF16Args & k, bool gateup, bool f32_out, unsigned blocks, hipStream_t s) {
    grouped_f16_launch<TQMOE_IQ3_S>(k, gateup, f32_out, blocks, s);
}
}  // namespace tqmoe
