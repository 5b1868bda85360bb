// Transfers from memory to LDS that pass no registers.
#pragma once
#include "common.cuh"

namespace tqmoe {
namespace {

// 16 bytes a lane from memory to LDS at `lds` (a wave-uniform byte address) + 16 * lane. The compiler does not count these:
// dma_wait() says when they are there.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 is a register the compiler reserves: what it keeps there itself must know of the write
__device__ __forceinline__ void dma16(const void * p, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(p), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
// all but the last N transfers of this wave are here (they finish in order); with BARRIER every wave's are
template <int N, bool BARRIER> __device__ __forceinline__ void dma_wait() {
    if constexpr (BARRIER) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "i"(N) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" :: "i"(N) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void * p) {
    return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint8_t *)(p)));
}

}  // namespace
}  // namespace tqmoe
