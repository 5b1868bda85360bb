// How the int8 grouped products put their integer sums and results into fp32 and fp16.
#pragma once
#include "common.cuh"
#include "decode_api.cuh"

namespace tqmoe {
namespace {

// Two paths that multiply the same rows must give them the same bits: the fold of a
// super-block and the epilogue are spelled with explicitly rounded operations, and the product that is converted to fp16
// passes through an opaque register, so that no path turns multiply + convert into one mixed-precision instruction
// (one rounding instead of two: different bits at ties).
__device__ __forceinline__ uint16_t to_half_bits(float v) {
    asm volatile("" : "+v"(v));
    return __half_as_ushort(__float2half_rn(v));
}
__device__ __forceinline__ uint16_t swiglu_half(float g_acc, float u_acc, float sc, const Glu glu) {
    float gv = __fmul_rn(g_acc, sc), uv = __fmul_rn(u_acc, sc);
    glu_clamp_inputs(glu, gv, uv);
    const float den = __fadd_rn(1.f, __expf(-gv));
    return to_half_bits(__fmul_rn(glu_clamp_silu(glu, __fdiv_rn(gv, den)), uv));
}
__device__ __forceinline__ uint16_t scaled_half(float acc, float sc, int bf16) {
    const float v = __fmul_rn(acc, sc);
    return bf16 ? float_to_bf16_bits(v) : to_half_bits(v);
}

}  // namespace
}  // namespace tqmoe
