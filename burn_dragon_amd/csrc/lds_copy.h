// Copies from memory straight into LDS (no registers in between), written out by hand.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

// Copies 16 bytes per lane from *src to LDS, the 64 lanes' pieces one after the other from dst (uniform over the
// wavefront).  Written out because the compiler waits for every copy that it knows of before any LDS read that might see
// it; the caller orders the two by its own wait (s_waitcnt vmcnt) and barrier.
// The LDS place travels in M0, which the compiler writes (it is an operand).  Between a scalar write of M0 and a load
// into LDS the hardware wants one wait state, and the compiler does not look for loads inside hand-written text: hence
// the s_nop, which costs nothing measurable beside the load.
typedef __attribute__((address_space(3))) void *bdh_lds_ptr_t;
__device__ __forceinline__ void bdh_copy_to_lds(const void *src, void *dst) {
  const unsigned int at = __builtin_amdgcn_readfirstlane((unsigned int)(uintptr_t)(bdh_lds_ptr_t)dst);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(at), "v"(src) : "memory");
}

// The same from base + offset bytes, base uniform over the wavefront: a loop that moves base along has no vector instructions
// for its addresses.
__device__ __forceinline__ void bdh_copy_to_lds(const void *base, unsigned int offset, void *dst) {
  const unsigned int at = __builtin_amdgcn_readfirstlane((unsigned int)(uintptr_t)(bdh_lds_ptr_t)dst);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(at), "v"(offset), "s"(base) : "memory");
}

// Waits until no more than `later` stages of COPIES copies each, issued by this wavefront after the stage that it needs, are
// still on their way (at most MOST of them are ever asked about).  Loads come back in the order of their issue.
template <int COPIES, int MOST>
__device__ __forceinline__ void bdh_wait_for_stage(int later) {
  if constexpr (MOST > 0) {
    if (later >= MOST) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COPIES * MOST) : "memory");
      return;
    }
    bdh_wait_for_stage<COPIES, MOST - 1>(later);
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}
