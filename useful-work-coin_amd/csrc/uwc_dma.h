// Building blocks of the kernels that feed int8 MFMAs from LDS tiles filled by DMA: LDS tile rows of
// P_BK = 128 bytes (one k step), 16-byte chunk c of row r at chunk c ^ ((r ^ (r >> 3)) & 7).
#pragma once
#include <type_traits>

#include "uwc_common.h"

#define P_BK 128
// lambdas are always inlined: an out-of-line call would take the accumulator arrays' addresses
#define P_AI __attribute__((always_inline))

namespace {

template <int I, int N, class F>
__device__ __forceinline__ void p_static_for_(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    p_static_for_<I + 1, N>(f);
  }
}
template <int N, class F>
__device__ __forceinline__ void p_static_for(F&& f) {
  p_static_for_<0, N>(f);
}

typedef void __attribute__((address_space(3)))* p_lptr_t;
typedef const v4i __attribute__((address_space(3)))* p_lds_v4i_t;

__device__ __forceinline__ u32 p_lds_addr(const u8* q) { return (u32)(uintptr_t)(p_lptr_t)q; }
__device__ __forceinline__ v4i p_lds(u32 a) { return *(p_lds_v4i_t)(uintptr_t)a; }
__device__ __forceinline__ int p_swz(int r) { return (r ^ (r >> 3)) & 7; }

// One wave-wide DMA: lane i's 16 bytes at sbase + voff land at LDS byte lds + 16 i (lds goes in
// M0). In asm so that the compiler's wait-count model does not see an LDS write in flight (it
// would then wait for every LDS read before each fragment use); the kernel waits on vmcnt and
// barriers itself before any stage is read, and refills a stage only after the barrier that ends
// every read of it.
__device__ __forceinline__ void p_dma(u32 voff, const void* sbase, u32 lds) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds) : "memory", "m0");
}

// p_dma with the non-temporal hint, for bytes read once: a weight that streams past the caches.
__device__ __forceinline__ void p_dma_nt(u32 voff, const void* sbase, u32 lds) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(voff), "s"(sbase), "s"(lds) : "memory", "m0");
}

// Wait until at most `younger` k steps of this wave's DMA (SEG instructions each) are in flight.
template <int SEG, int MAXY>
__device__ __forceinline__ void p_wait_vm(int younger) {
  static_assert(MAXY * SEG < 64, "vmcnt is 6 bits");
  if (MAXY >= 3 && younger >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * SEG) : "memory");
  else if (MAXY >= 2 && younger >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * SEG) : "memory");
  else if (MAXY >= 1 && younger >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SEG) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// A TB x TB MFMA block of int8: PASSES of a 128-byte k step, lane l holding row l % TB and 16-byte
// chunk 8 / PASSES kp + l / TB of an operand in pass kp, and, of the transposed product, row l % TB with the
// 16-byte pieces (four columns) 2 g + l / 32 (TB = 32, g < 4) or l / 16 (TB = 16).
template <int TB>
struct Mfma;
template <>
struct Mfma<32> {
  typedef v16i acc_t;
  static constexpr int PASSES = 4, G = 4;
  static __device__ __forceinline__ v16i mul(v4i b, v4i a, v16i c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(b, a, c, 0, 0, 0); }
};
template <>
struct Mfma<16> {
  typedef v4i acc_t;
  static constexpr int PASSES = 2, G = 1;
  static __device__ __forceinline__ v4i mul(v4i b, v4i a, v4i c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a, c, 0, 0, 0); }
};

}  // namespace
