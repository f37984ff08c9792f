// Direct loads into LDS, in rings of steps: what the tiled products share.
#pragma once
#include "sp_common.h"

namespace sp {

// 16 bytes per lane from base + off to lds + 16 lane, without a register on the way.  (The builtin of the same makes every later read of
// LDS wait for it.  m0 is named, so that no value another instruction needs in it is carried past; the compiler calls that reserved.)
// ONCE: past the L2's other lines.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool ONCE>
__device__ __forceinline__ void ring_load(uint32_t off, const char* base, uint32_t lds) {
  if constexpr (ONCE)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// Waits until at most min(later, MOST) steps of L loads each are on their way, and for this wave's reads of LDS
template <int L, int MOST>
__device__ __forceinline__ void ring_wait(int later) {
  if constexpr (MOST == 0) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  } else {
    if (later >= MOST) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(L* MOST) : "memory");
    else ring_wait<L, MOST - 1>(later);
  }
}

__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ uint32_t lds_address(const char* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }

}  // namespace sp
