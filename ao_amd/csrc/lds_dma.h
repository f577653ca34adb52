// Direct loads, global memory -> LDS, 16 or 4 bytes a lane: lane L of the wave lands at lds + at + 16 L (4 L), `at` a constant, so that
// the LDS address goes into m0 by one instruction.
#pragma once
#include "common.h"

namespace ao {

// from a scalar base and a 32-bit byte offset of each lane
__device__ __forceinline__ void lds_dma16(uint32_t lds, int at, const void* base, uint32_t off) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds), "i"(at) : "memory", "scc");
}
__device__ __forceinline__ void lds_dma4(uint32_t lds, int at, const void* base, uint32_t off) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "s"(lds), "i"(at) : "memory", "scc");
}
// from each lane's own address
__device__ __forceinline__ void lds_dma16(uint32_t lds, int at, const void* p) {
    asm volatile("s_add_u32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"((uint64_t)(uintptr_t)p), "s"(lds), "i"(at) : "memory", "scc");
}
__device__ __forceinline__ void lds_dma4(uint32_t lds, int at, const void* p) {
    asm volatile("s_add_u32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"((uint64_t)(uintptr_t)p), "s"(lds), "i"(at) : "memory", "scc");
}

}  // namespace ao
