// Building blocks of the walks that are laid out by hand: loops unrolled over compile-time indices, LDS accesses by byte address,
// products into accumulation registers, waits that count.
#pragma once
#include <utility>
#include "nsa_common.hpp"

namespace nsa {

typedef __attribute__((__vector_size__(4 * sizeof(int)))) int rsrc4;

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) { static_for_impl(f, std::make_integer_sequence<int, N>{}); }

// c += a b with c in accumulation registers.  The compiler does not see the instruction: operands written by vector instructions need
// two wait states (FRESH), and the accumulators are read only behind the loop.
template <bool FRESH>
__device__ __forceinline__ void mfma32_acc(floatx16& c, const bf16x8& a, const bf16x8& b) {
  if (FRESH) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
typedef __attribute__((address_space(1))) bf16x8* glb_x8;
typedef __attribute__((address_space(3))) bf16x8* lds_x8;
typedef __attribute__((address_space(3))) bf16x4* lds_x4;
typedef __attribute__((address_space(3))) shortx4* lds_s4;
typedef __attribute__((address_space(3))) floatx4* lds_f4;
typedef __attribute__((address_space(3))) int* lds_i;
__device__ __forceinline__ bf16x8 lds_read8(unsigned a) { return *(lds_x8)a; }
__device__ __forceinline__ bf16x8 lds_read8_tr(unsigned a, unsigned a2) {
  const shortx4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)a), y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)a2);
  typedef __attribute__((__vector_size__(8 * sizeof(short)))) short shortx8;
  shortx8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) { r[i] = x[i]; r[4 + i] = y[i]; }
  return __builtin_bit_cast(bf16x8, r);
}
// nothing derived from x is moved across this
__device__ __forceinline__ void opaque(unsigned& x) { asm volatile("" : "+v"(x)); }
template <int N>
__device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

}  // namespace nsa
