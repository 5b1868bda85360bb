// Decode-sized products of IQ4_XS banks (decode_mfma_kernels.cuh); every shape the entry points let through fits the kernel.
#include "decode_mfma_kernels.cuh"

namespace tqmoe {

template <> void DecodeLaunch<TQMOE_IQ4_XS>::matvec(Split, int nb, const MatvecArgs & k, hipStream_t s) {
    mfma_launch<TQMOE_IQ4_XS>(nb, k.b0, k.b1, k.image, k.y0, k.y1, k.ytype, k.ids, k.A, k.xdiv, k.mode, k.slots, k.topk, k.shared_cols, 0, false, Glu{0.f, 0}, s);
}
template <> void DecodeLaunch<TQMOE_IQ4_XS>::gateup(Split, const GateupArgs & k, hipStream_t s) {
    mfma_launch<TQMOE_IQ4_XS>(2, k.bg, k.bu, k.ximage, k.aimage, nullptr, TQMOE_F32, k.ids, k.A, k.slots, k.mode, k.slots, k.topk, k.shared_ff, 1, true, k.glu, s, k.route);
}
template <> void DecodeLaunch<TQMOE_IQ4_XS>::down_combine(const DownCombineArgs & k, hipStream_t s) { down_combine_launch<TQMOE_IQ4_XS>(k, s); }

}  // namespace tqmoe
