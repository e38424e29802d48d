// LDS staging: DMA from global memory, and the order of rows that are read as MFMA
// operands. The DMA is asm since the compiler otherwise makes LDS reads wait for
// DMAs into other parts of a ring (and drains all of them).
#pragma once
#include "qvex_common.h"

namespace {

// One DMA of 16 (4) bytes per lane: lane l lands at lds + 16 l (lds + 4 l). It
// has no register outputs; nothing reads the bytes before arrive().
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
               : "memory", "m0");
}
__device__ __forceinline__ void dma16_nt(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds), "v"(off), "s"(base)
               : "memory", "m0");
}
__device__ __forceinline__ void dma4(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base)
               : "memory", "m0");
}

// At most N of this wave's DMAs still in flight, its LDS reads done, and every
// wave of the block here. The builtin (LDS reads only) tells the compiler that
// they are done: it would otherwise wait for them again behind later ones.
template <int N>
__device__ __forceinline__ void arrive() {
  __builtin_amdgcn_s_waitcnt(0xc07f);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

__device__ __forceinline__ uint32_t lds_offset(void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)p;
}

// Rows of 256 bytes in LDS with their 16-byte chunk ch at ch ^ row_swizzle(row): the 16
// lanes that one pass of ds_read_b128 serves (0-3, 12-15 of one quarter, 4-11 of the
// next) then hit 16 different bank groups.
__device__ __forceinline__ int row_swizzle(int r) {
  const int b = (r >> 2) & 3;                                   // b -> 0, 2, 3, 1
  return ((((b << 1) & 3) ^ ((b >> 1) * 3)) << 2) | (r & 3);
}

}  // namespace
