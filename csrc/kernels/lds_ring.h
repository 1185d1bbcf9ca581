// Memory to LDS in pieces of 1 KB, through a ring of tiles of a wave's own: no barrier, a wave waits for its own pieces.
// Whole runs that are marked as read once come at 6.8 TB/s, 64 bytes of 16 rows a load (MFMA fragments) at 5.8 to 6.3.
// In asm, so that hipcc orders nothing behind the pieces and counts none of them: a load that it knows of, in flight beside
// them, makes it wait for all.  M0 is kept.
#pragma once
#include "common.h"

namespace {

typedef __attribute__((address_space(3))) void ring_lds_t;

__device__ __forceinline__ uint32_t lds_at(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(ring_lds_t*)p);
}

// lane l's 16 bytes of sbase + voff land at lds_addr + 16 l
template <bool NT>
__device__ __forceinline__ void ring_piece(uint32_t voff, const void* sbase, uint32_t lds_addr) {
  unsigned keep;
  if constexpr (NT)
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
        : "=&s"(keep) : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
  else
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
        : "=&s"(keep) : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}

// each lane's 16 bytes from a place of its own
__device__ __forceinline__ void ring_piece_at(const void* src, uint32_t lds_addr) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(src), "s"(lds_addr) : "memory");
}

// each lane's 4 bytes, to lds_addr + 4 l
__device__ __forceinline__ void ring_word_at(const void* src, uint32_t lds_addr) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(src), "s"(lds_addr) : "memory");
}

template <int N>
__device__ __forceinline__ void ring_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(N) : "memory");
}

// behind tile j of `tiles` (NP pieces each, T of them asked for ahead): those that are asked for
template <int T, int NP>
__device__ __forceinline__ void ring_landed(int j, int tiles) {
  static_assert(T >= 2 && T <= 4 && NP * (T - 1) <= 63, "");
  const int left = tiles - 1 - j;
  if (left >= T - 1) ring_wait<NP * (T - 1)>();
  else if (T > 3 && left == 2) ring_wait<2 * NP>();
  else if (T > 2 && left == 1) ring_wait<NP>();
  else ring_wait<0>();
}

}  // namespace
