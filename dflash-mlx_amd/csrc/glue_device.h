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

// sigmoid(x) of an x that a 16-bit array holds, with the error of 1 / (1 + expf(-x)) in 14 vector instructions for its 30.
//  * -x log2(e) is n + f, n its nearest integer (left in the low bits of a sum with 1.5 2^23).  kLog2E has 13 bits, so that with the
//    at most 11 of x its product is exact, and so is the difference to n: f is rounded once.
//  * 2^n is made of n's bits, and 1 + 2^f 2^n is one fma, kept times 2^-24: its reciprocal is a normal number for every x,
//    and what comes out is rounded once more only where it is a subnormal one.  x is bounded where the result is 1 or
//    less than any number above 0; the bounds let a NaN pass.
//  * a Newton step takes the hardware's reciprocal from one unit to the nearest number but for rare ties.
// Over all numbers of a type, against 64 bits, largest and root mean square relative error: bf16 1.18e-7 and 1.51e-8, fp16 1.20e-7 and
// 3.41e-8, of either form; 1 / (1 + expf(-x)) has 0 below x = -88.7, where this still has the subnormal numbers.  Conv and gates of
// 1024 tokens of 16 + 16 + 32 heads of 128 18.6 -> 16.2 us, a block of 16 of them with its recurrence 16.9 -> 16.3 us.
__device__ __forceinline__ float sigmoid_of_half(float x) {
  constexpr float kLog2E = 5909.f / 4096.f, kRest = 6.8087763963407e-5f, kRound = 0x1.8p23f, kScale = 0x1p-24f;
  const float u = __builtin_elementwise_maximum(__builtin_elementwise_minimum(-x, 104.f), -30.f);
  const float m = __builtin_fmaf(u, kLog2E, kRound), n = m - kRound;
  const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(u, kRest, __builtin_fmaf(u, kLog2E, -n)));
  const float d = __builtin_fmaf(e, __uint_as_float((__float_as_uint(m) << 23) + __float_as_uint(kScale)), kScale);
  const float r = __builtin_amdgcn_rcpf(d);
  return kScale * __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}

// sigmoid(x), for an array of type dt
__device__ __forceinline__ float sigmoid_for(float x, int dt) {
  return dt == DFLASH_FP32 ? 1.0f / (1.0f + expf(-x)) : sigmoid_of_half(x);
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
  if (dt == DFLASH_BF16 && PER % 2 == 0) {  // two elements to a conversion
    typedef __attribute__((ext_vector_type(2))) __bf16 pair_t;
    typedef __attribute__((ext_vector_type(2))) float floats_t;
    uint32_t words[PER];
#pragma unroll
    for (int e = 0; e + 1 < PER; e += 2) words[e / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((floats_t{v[e], v[e + 1]}), pair_t));
    uint16_t* const dst = (uint16_t*)p + i;
#pragma unroll
    for (int e = 0; e + 1 < PER; e += PER % 4 == 0 ? 4 : 2) {
      if constexpr (PER % 4 == 0) *reinterpret_cast<uint2*>(dst + e) = uint2{words[e / 2], words[e / 2 + 1]};
      else *reinterpret_cast<uint32_t*>(dst + e) = words[e / 2];
    }
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

// PER adjacent 16-bit elements stored as load_adjacent_raw() left them.
template <int PER>
__device__ __forceinline__ void store_raw(uint16_t* dst, const uint32_t (&raw)[PER]) {
  if constexpr (PER == 4) {
    *reinterpret_cast<uint2*>(dst) = make_uint2(raw[0], raw[1]);
  } else if constexpr (PER == 2) {
    *reinterpret_cast<uint32_t*>(dst) = raw[0];
  } else {
#pragma unroll
    for (int e = 0; e < PER; ++e) dst[e] = (uint16_t)raw[e];
  }
}

// A number of 32 bits that is one before it is rounded to fp16: the compiler makes one instruction with one rounding
// (v_fma_mixlo_f16) of some products and their conversion, where it knows the type, and not of others.
__device__ __forceinline__ float in_full(float v) {
  asm("" : "+v"(v));
  return v;
}

// Norm and rotation of one head by a wave, a lane on PER adjacent features: x <- turned(round(x rsqrt(mean x^2 + eps) w)), the
// products and sums of the rotation rounded one by one, as the array operators do it.  other: the lane of the pair's other half.
template <int PER>
__device__ __forceinline__ void norm_and_turn(float (&x)[PER], const float (&w)[PER], float eps, const float (&cs)[PER],
                                              const float (&sn)[PER], bool rotates, bool upper, int other, int dt) {
#pragma clang fp contract(off)
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < PER; ++e) ss += x[e] * x[e];
  // (the array operators divide by a number by multiplying with its reciprocal)
  const float inv_rms = 1.0f / sqrtf(wave_sum(ss) * (1.0f / (float)(64 * PER)) + eps);
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    x[e] = round_through(in_full(x[e] * inv_rms * w[e]), dt);
    const float y = __shfl(x[e], other, 64);  // the other half's feature of the pair
    if (rotates) {
      const float a = x[e] * cs[e], d = y * sn[e];
      x[e] = in_full(upper ? d + a : a - d);
    }
  }
}

}  // namespace
}  // namespace dflash
