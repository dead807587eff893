// mh_dma.cuh — memory to LDS without a register in between
// (global_load_lds): lane i's piece lands at lds + 16 i (or 4 i), lds uniform
// across the wave.
//
// The compiler does not see these loads: with the builtin it makes every LDS
// read wait for all of them, which ends the pipelining that they are for. So
// a kernel that uses them counts them itself: dma_wait<LEFT> holds the wave
// until all but its last LEFT vector memory operations are done (they
// complete in issue order; others that the compiler puts among them only
// make the wait longer), and dma_barrier then makes every wave's visible. A
// buffer is loaded again only after a barrier that follows its last reads,
// and the last loads are waited for before the block ends.
//
// The LDS address is in m0, which the loads take as an operand: the compiler
// sets it, and knows of every value that it holds (a statement that wrote m0
// itself would change it behind the compiler's back, and naming a reserved
// register as clobbered does not keep a value across it).
#pragma once

#include "mh_internal.h"

namespace mh {

__device__ __forceinline__ uint32_t lds_offset(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t *)p;
}
__device__ __forceinline__ void dma16(uint32_t lds, const uint8_t *p) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(p) : "memory");
}
__device__ __forceinline__ void dma4(uint32_t lds, const uint8_t *p) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %1, off" ::"{m0}"(lds), "v"(p) : "memory");
}
__device__ __forceinline__ uint64_t uniform_addr(const uint8_t *p) {
    const uint64_t a = (uint64_t)p;
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a) |
           (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32)) << 32;
}
// (from a scalar base and 32-bit lane offsets: half the address registers. Five
// wait states before the load: its scalar operands may come from a vector
// instruction, and the compiler cannot see that it reads them.)
__device__ __forceinline__ void dma16(uint32_t lds, const uint8_t *base, uint32_t off) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(__builtin_amdgcn_readfirstlane(lds)),
                 "v"(off), "s"(uniform_addr(base))
                 : "memory");
}
__device__ __forceinline__ void dma4(uint32_t lds, const uint8_t *base, uint32_t off) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dword %1, %2" ::"{m0}"(__builtin_amdgcn_readfirstlane(lds)),
                 "v"(off), "s"(uniform_addr(base))
                 : "memory");
}
template <int LEFT>
__device__ __forceinline__ void dma_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}
// (this wave's LDS reads are done first: their buffer may be loaded next)
__device__ __forceinline__ void dma_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace mh
