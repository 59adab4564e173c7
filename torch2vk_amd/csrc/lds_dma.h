// Stages of a tile brought straight from global memory into LDS, for the kernels that run their loops on it.
#pragma once

#include "common.h"

namespace t2h {

// LDS-DMA of 16 B per lane into lds_addr + 16 * lane.  M0 holds the LDS base; one wait state separates its
// write from the load that reads it.
__device__ __forceinline__ void lds_dma16(const void* g, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_addr)
                 : "memory", "m0");
}

// s_waitcnt of the global counter alone (its 6 bits are split over the immediate), and of the LDS counter alone
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N < 64, "6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (3 << 14)); }

// A barrier that waits for nothing but the other waves: the loads in flight are the caller's to wait for.
__device__ __forceinline__ void wave_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

}  // namespace t2h
