// A wavefront's copy of 1024 bytes from memory to LDS that the compiler does not count among its loads: whoever asks for one waits for it himself.
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

namespace shainet {

// Lane l's 16 bytes at base + offset (its own) go to lds + 16 l.  nt: read once.  (M0 holds the place in LDS.  The compiler keeps it out of its
// register allocation, of which it warns, but sets it itself for other instructions and has to know that it is another one behind this.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool NT>
__device__ __forceinline__ void copy_to_lds(void *lds, const void *base, unsigned offset) {
  const unsigned to = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)lds);
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" : : "s"(to), "v"(offset), "s"(base) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(to), "v"(offset), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

}  // namespace shainet
