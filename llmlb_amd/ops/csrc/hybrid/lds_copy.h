// Copies from global memory straight to LDS: a wave moves 1 KB per
// instruction without registers, and waits for them by count.
#pragma once
#include "common.h"

// where lanes read that have nothing to copy
static __device__ __align__(16) unsigned zero_piece[4];

// 64 lanes copy 16 bytes each from their own addresses to 1 KB of LDS from
// byte ``to`` on.  The copy counts as a load of the wave; nothing but
// an explicit wait waits for it.
__device__ __forceinline__ void copy_to_lds(const bf16_t* src, unsigned to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(src)
               : "memory");
}
// the same from ``at`` bytes behind one address of the wave's
__device__ __forceinline__ void copy_to_lds(const bf16_t* base, unsigned at,
                                            unsigned to) {
  const unsigned long long b = (unsigned long long)base;
  const unsigned long long wave_base =
      (unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(b >> 32))
          << 32 |
      (unsigned)__builtin_amdgcn_readfirstlane((unsigned)b);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(at),
                 "s"(wave_base)
               : "memory");
}
// 64 lanes copy four bytes each to 256 bytes of LDS
__device__ __forceinline__ void copy_words_to_lds(const int* src,
                                                  unsigned to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
               ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(src)
               : "memory");
}
// the same as the first for data that nobody reads again
__device__ __forceinline__ void stream_to_lds(const bf16_t* src,
                                              unsigned to) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt"
      ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(src)
      : "memory");
}
__device__ __forceinline__ unsigned lds_byte(const void* p) {
  return (unsigned)(uintptr_t)((const __attribute__((address_space(3))) char*)p);
}
// All but the newest N copies and loads of the wave are done.
template <int N>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// ... and its LDS reads; then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N)
               : "memory");
}
