// Loads from memory straight into LDS, for kernels that stream weights past a few rows.
#pragma once
#include "common.h"

namespace lipa {

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __amdgpu_buffer_rsrc_t rsrc;

__device__ __forceinline__ rsrc window(const void* base) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p), hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0, 0xFFFFFFFFu, 0x00020000);
}
// 64 lanes x 16 bytes from memory into LDS [dst, dst + 1 KB), lane after lane; M0 is put back
#define LIPA_TO_LDS(HINT)                                                                                   \
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen" HINT \
               " lds\n\ts_mov_b32 m0, %0"                                                                   \
               : "=&s"(keep)                                                                                \
               : "s"(dst), "v"(voff), "s"(rs), "s"(soff)                                                    \
               : "memory")
__device__ __forceinline__ void to_lds(const rsrc& rs, uint32_t dst, uint32_t voff, uint32_t soff) {
  uint32_t keep;
  LIPA_TO_LDS("");
}
// ... of bytes that nobody else reads in this launch (a weight's rows, each in one workgroup): what they would push out of the caches stays
__device__ __forceinline__ void to_lds_once(const rsrc& rs, uint32_t dst, uint32_t voff, uint32_t soff) {
  uint32_t keep;
  LIPA_TO_LDS(" nt");
}
#undef LIPA_TO_LDS
// until all but the last `left` units (at most R), of D loads each, have landed
template <int D, int R>
__device__ __forceinline__ void wait_units(int left) {
  if constexpr (R == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    if (left >= R)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R * D) : "memory");
    else
      wait_units<D, R - 1>(left);
  }
}

}  // namespace lipa
