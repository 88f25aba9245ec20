// Device helpers of the layer-glue kernels (gdn_glue.hip, attn_glue.hip): a wave on one head, a lane on
// PER = D / 64 adjacent elements of it.
#pragma once

#include "dflash_common.h"

namespace dflash {
namespace {

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// sigmoid(x), for an array of type dt.  16-bit arrays take the hardware's exp2 and reciprocal (each within an ulp of fp32, where
// half a unit of the result is 2^-9 or 2^-12 of it): 4 instructions for about 30, of what the kernels here spend most on.
__device__ __forceinline__ float sigmoid_for(float x, int dt) {
  return dt == DFLASH_FP32 ? 1.0f / (1.0f + expf(-x)) : __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * x));
}

// x * sigmoid(x) with the sigmoid and the product each rounded to the array dtype
__device__ __forceinline__ float silu_rounded(float x, int dt) {
  return round_through(x * round_through(sigmoid_for(x, dt), dt), dt);
}

// PER adjacent elements of an array, starting at element i (a multiple of PER), as raw bits
// (16-bit types zero-extended): 2-byte types in 64-bit accesses when PER is a multiple of 4, one
// 32-bit access for a pair.  Loading and interpreting are separate steps so that a wave can have
// all of its requests out before it waits for the first answer: with the dtype switch inside, every
// load sits in a branch of its own together with its conversion and is awaited there.
template <int PER>
__device__ __forceinline__ void load_adjacent_raw(const void* p, size_t i, bool wide, uint32_t (&raw)[PER]) {
  // no arithmetic on what comes back: the words stay as loaded (two elements per word for an even
  // number of 16-bit elements) until unpack_adjacent()
  if (wide) {
    const uint32_t* src = (const uint32_t*)p + i;
#pragma unroll
    for (int e = 0; e < PER; ++e) raw[e] = src[e];
  } else if (PER % 4 == 0) {
#pragma unroll
    for (int e = 0; e < PER; e += 4) {
      const uint2 w = *reinterpret_cast<const uint2*>((const uint16_t*)p + i + e);
      raw[e / 2] = w.x, raw[e / 2 + 1 < PER ? e / 2 + 1 : 0] = w.y;
    }
  } else if (PER == 2) {
    raw[0] = *reinterpret_cast<const uint32_t*>((const uint16_t*)p + i);
  } else {
#pragma unroll
    for (int e = 0; e < PER; ++e) raw[e] = ((const uint16_t*)p)[i + e];
  }
}
__device__ __forceinline__ float bits_as_f32(uint32_t bits, int dt) {
  return dt == DFLASH_BF16 ? bf16_bits_to_f32(bits) : dt == DFLASH_FP16 ? f16_bits_to_f32(bits) : __uint_as_float(bits);
}
template <int PER>
__device__ __forceinline__ void unpack_adjacent(const uint32_t (&raw)[PER], int dt, float (&out)[PER]) {
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    constexpr bool kPacked = PER % 4 == 0 || PER == 2;  // as load_adjacent_raw() packs 16-bit elements
    if (dt == DFLASH_FP32 || !kPacked) {
      out[e] = bits_as_f32(raw[e], dt);
    } else {
      out[e] = bits_as_f32((e & 1) ? raw[e / 2] >> 16 : raw[e / 2] & 0xFFFFu, dt);
    }
  }
}
__device__ __forceinline__ uint32_t load_one(const void* p, size_t i, bool wide) {
  if (wide) return ((const uint32_t*)p)[i];
  return ((const uint16_t*)p)[i];
}
template <int PER>
__device__ __forceinline__ void load_adjacent(const void* p, size_t i, int dt, float (&out)[PER]) {
  uint32_t raw[PER];
  load_adjacent_raw<PER>(p, i, dt == DFLASH_FP32, raw);
  unpack_adjacent<PER>(raw, dt, out);
}
// PER adjacent elements stored from fp32 (round to nearest even), packed like the loads.
template <int PER>
__device__ __forceinline__ void store_adjacent(void* p, size_t i, int dt, const float (&v)[PER]) {
  if (dt == DFLASH_FP32) {
    float* dst = (float*)p + i;
#pragma unroll
    for (int e = 0; e < PER; ++e) dst[e] = v[e];
    return;
  }
  uint32_t h[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) h[e] = dt == DFLASH_BF16 ? f32_to_bf16_bits(v[e]) : f32_to_f16_bits(v[e]);
  if (PER % 4 == 0) {
#pragma unroll
    for (int e = 0; e < PER; e += 4)
      *reinterpret_cast<uint2*>((uint16_t*)p + i + e) =
          uint2{h[e] | (h[e + 1 < PER ? e + 1 : 0] << 16), h[e + 2 < PER ? e + 2 : 0] | (h[e + 3 < PER ? e + 3 : 0] << 16)};
  } else if (PER == 2) {
    *reinterpret_cast<uint32_t*>((uint16_t*)p + i) = h[0] | (h[PER > 1 ? 1 : 0] << 16);
  } else {
#pragma unroll
    for (int e = 0; e < PER; ++e) ((uint16_t*)p)[i + e] = (uint16_t)h[e];
  }
}

}  // namespace
}  // namespace dflash
