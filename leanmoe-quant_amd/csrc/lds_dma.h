// Direct loads from global memory to LDS, and the LDS addresses they take.
//
// asm, because the compiler drains every direct load (vmcnt 0) before any LDS
// read: the caller waits for its own.  m0 holds the LDS address of lane 0, lane
// l's element follows at l times its size; the asm writes m0 and says so.
#pragma once

#include "common.h"

// LDS byte address of a shared array (also marks the array as written by the
// direct loads' asm, which the compiler cannot see into).
typedef __attribute__((address_space(3))) uint8_t lds_byte;
__device__ __forceinline__ uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const lds_byte*)p; }

// The clobber makes the compiler write m0 again before any use of its own; that m0 is
// a register it never allocates is what -Winline-asm warns of.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 64 lanes x 16 bytes from base + off (per lane), or from addr, to LDS at `to` + 16 lane.
__device__ __forceinline__ void dma16(uint32_t to, uint32_t off, const uint8_t* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(to), "v"(off), "s"(base)
               : "m0", "memory");
}
__device__ __forceinline__ void dma16(uint32_t to, uint64_t addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(to), "v"(addr)
               : "m0", "memory");
}
// 64 lanes x 2 bytes from addr (per lane), zero-extended, to LDS at `to` + 4 lane.
__device__ __forceinline__ void dma2(uint32_t to, uint64_t addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, off"
               :
               : "s"(to), "v"(addr)
               : "m0", "memory");
}
#pragma clang diagnostic pop
