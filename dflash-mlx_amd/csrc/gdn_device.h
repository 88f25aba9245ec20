// Shared by the GatedDeltaNet kernels: fp32 values as sums of bf16 pieces for the matrix cores.
#pragma once

#include "dflash_common.h"

namespace dflash {
// ---- exact products on the 16-bit matrix cores ---------------------------------------------
// An fp32 value is the sum of three bf16 values (its leading 8 significant bits, the next 8 of
// what is left, and the rest: 24 bits in all, each piece cut off, not rounded, so every
// difference is exact), and a bf16 times a bf16 is exact in fp32.  A product of an fp32 matrix
// with a matrix whose entries are bf16 numbers can therefore run as three passes of
// v_mfma_f32_16x16x32_bf16 (9 ns for 32 steps of the sum) instead of eight of
// v_mfma_f32_16x16x4_f32 (16 ns for 4 steps): the same products, summed in fp32 in another order.
// the upper halves of a and b (a in the low half): two bf16 numbers, cut off
__device__ __forceinline__ uint32_t upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float below_bf16(float v) {  // v minus its leading 8 significant bits
  return v - __uint_as_float(__float_as_uint(v) & 0xffff0000u);
}
template <int N>
struct Pieces {  // three bf16 pieces of N fp32 values, packed in pairs
  uint32_t hi[N / 2], mid[N / 2], lo[N / 2];
};
template <int N>
__device__ __forceinline__ Pieces<N> split_bf16(const float (&f)[N]) {
  Pieces<N> p;
  float r1[N], r2[N];
#pragma unroll
  for (int j = 0; j < N; ++j) r1[j] = below_bf16(f[j]), r2[j] = below_bf16(r1[j]);
#pragma unroll
  for (int j = 0; j < N / 2; ++j) {
    p.hi[j] = upper_halves(f[2 * j], f[2 * j + 1]);
    p.mid[j] = upper_halves(r1[2 * j], r1[2 * j + 1]);
    p.lo[j] = upper_halves(r2[2 * j], r2[2 * j + 1]);
  }
  return p;
}
}  // namespace dflash
