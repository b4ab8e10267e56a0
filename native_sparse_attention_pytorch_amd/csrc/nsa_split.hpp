// fp32 products on the bf16 matrix instructions: every fp32 operand is the sum of three bf16 numbers (8 + 8 + 8 bits of
// significand, exact; the first is the operand cut off, so that nothing rounds up to infinity), and of the nine products of two
// operands' parts only that of both third parts, 2^-32 of the product, is left out.  The eight cost half of the fp32 matrix
// instructions' time.  The products of the leading parts and the seven small ones are summed in accumulators of their own, so a single
// product is rounded as an fp32 multiplication is, and a sum once per 16 products.  Error against float64 in units of fp32 fused
// multiply-adds', rms and largest: sums of 1 product 1.00 / 1.01, 2 0.82 / 1.17, 4 0.66 / 0.88, 16 0.43 / 0.39, 1024 0.32 / 0.36.  (Six products, without
// the two of a second and a third part: 1 1.34 / 4.0, 2 1.11 / 2.0, 4 0.87 / 0.95, and the projections' time 0.83 of the eight's.)
// That holds for operands above 2^-110.  Below, the third part leaves the range of bf16 and an operand is kept to 2^-134: a sum
// whose operands are all that small loses digits (at 2^-120 it is 7e-6 off), beside larger ones nothing is seen of it.
#pragma once
#include "nsa_common.hpp"

namespace nsa {

struct Split3 { bf16x4 part[3]; };

__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  bf16x2 r;
  r[0] = (__bf16)a;
  r[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, r);
}

// An infinity or NaN is its own leading part and makes the second one NaN: the sums of small products mean nothing then, and
// split_sum() takes those of leading products alone.
__device__ __forceinline__ void split2(float x0, float x1, uint32_t (&part)[3]) {
  const uint32_t u0 = __builtin_bit_cast(uint32_t, x0), u1 = __builtin_bit_cast(uint32_t, x1);
  part[0] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
  const float r0 = x0 - __builtin_bit_cast(float, u0 & 0xffff0000u), r1 = x1 - __builtin_bit_cast(float, u1 & 0xffff0000u);
  part[1] = bf16_pair(r0, r1);
  part[2] = bf16_pair(r0 - __builtin_bit_cast(float, part[1] << 16), r1 - __builtin_bit_cast(float, part[1] & 0xffff0000u));
}

__device__ __forceinline__ Split3 split4(floatx4 x) {
  uint32_t a[3], b[3];
  split2(x[0], x[1], a);
  split2(x[2], x[3], b);
  Split3 s;
#pragma unroll
  for (int p = 0; p < 3; ++p) s.part[p] = __builtin_bit_cast(bf16x4, uintx2{a[p], b[p]});
  return s;
}

// sums of leading and of small products -> the product
__device__ __forceinline__ float split_sum(float lead, float small) { return fabsf(lead) < INFINITY ? lead + small : lead; }

}  // namespace nsa
