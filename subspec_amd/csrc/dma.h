// Copies from memory straight into LDS, waited for by hand: the compiler waits for every LDS copy that it knows of before any
// LDS read, so the requests are inline assembly and the kernels that use them place their own waits.  (s_nop: the wait state that
// M0 needs before a copy reads it.  The base must have been in scalar registers for five wait states: see dense_tile_kernel.)
#pragma once
#include "common.h"

namespace subspec {

// 16 bytes per lane from base + voffset into LDS (lds_base + 16 * lane); NT: as streaming data
template <bool NT>
__device__ __forceinline__ void dma16(uint32_t lds_base, uint32_t voffset, const void* base) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_base), "v"(voffset), "s"(base) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(voffset), "s"(base) : "memory", "m0");
}
// a wavefront-uniform address in scalar registers
__device__ __forceinline__ const uint8_t* uniform_ptr(const uint8_t* p) {
  const uint64_t a = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return (const uint8_t*)(uintptr_t)((uint64_t)hi << 32 | lo);
}
template <int N> __device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

}  // namespace subspec
