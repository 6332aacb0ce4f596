// Direct global -> LDS loads, shared by the GEMM kernels.
#pragma once

#include "wm_common.h"

namespace wm {

// Lane i writes LDS address lds + size * i. Written as inline assembly so the compiler does
// not treat them as LDS stores it must wait for before every LDS read (it cannot tell a
// ring's stages apart); a K loop's explicit vmcnt waits and barriers order them instead. M0
// carries the wave-uniform LDS address (nothing else in these kernels uses M0); an M0 write
// needs wait states before an LDS DMA reads it.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
}
// The global address is a wave-uniform base in scalar registers plus a 32-bit per-lane
// offset, so no 64-bit addresses occupy vector registers.
// NT: with the non-temporal hint, for lines read once per call.
template <bool NT = false>
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds), "v"(off), "s"(base)
                 : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
                 : "memory");
}
__device__ __forceinline__ void dma4(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base)
               : "memory");
}

}  // namespace wm
