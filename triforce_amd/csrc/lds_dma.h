// LDS-DMA that the compiler does not count, the meetings of a workgroup that go with it, and the wait behind products in inline asm, which it does not
// guard.  Behind its own form of the DMA it waits for all reads of LDS that are under way wherever one is needed.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// 16 bytes a lane from `from` + off to LDS at `at` + 16 * lane (`at` the same in all lanes).
__device__ __forceinline__ void lds_dma(uint32_t at, uint32_t off, const void* from) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(at), "v"(off), "s"(from) : "memory", "m0");
}
// All waves are here and all but the LEFT youngest of this one's loads have landed; READS: its LDS accesses are done too.  No access crosses.
template <int LEFT, bool READS> __device__ __forceinline__ void meet_dma() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((READS ? 0x0070 : 0x0F70) | (LEFT & 15) | (LEFT >> 4 << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// Twelve wait states between products and what else touches their sums: behind a 16 x 16 x 32 product (eight passes) eleven are needed.
__device__ __forceinline__ void hold_sums() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 11" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
