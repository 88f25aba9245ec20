// A GatedDeltaNet block as its projections leave it: the conv, the activation, the norms and the gates of
// gdn_glue.hip's prepare kernel, for kernels that go on with the recurrence themselves (bf16 arrays, four taps).  Operator for
// operator and sum for sum as there, so that both ways give the same bits.
#pragma once

#include "glue_device.h"

namespace dflash {
namespace {

// v + (v of the lane that the DPP control names)
template <int CTRL>
__device__ __forceinline__ float plus_dpp(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// v summed over the lanes that differ in bits 4 and 5 (16 and 32 apart)
__device__ __forceinline__ float plus_far(float v, bool both) {
  const auto near = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(near[0]) + __uint_as_float(near[1]);
  if (!both) return v;
  const auto far = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(far[0]) + __uint_as_float(far[1]);
}
// v summed over LANES adjacent lanes, neighbours first: the sums of a butterfly of shuffles, which took the LDS five answers one after the other
// (quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror, row_mirror, then swaps of rows of 16 lanes).
template <int LANES>
__device__ __forceinline__ float sum_over_lanes(float v) {
  if constexpr (LANES >= 2) v = plus_dpp<0xB1>(v);
  if constexpr (LANES >= 4) v = plus_dpp<0x4E>(v);
  if constexpr (LANES >= 8) v = plus_dpp<0x141>(v);
  if constexpr (LANES >= 16) v = plus_dpp<0x140>(v);
  if constexpr (LANES >= 32) v = plus_far(v, LANES >= 64);
  return v;
}

// Sum of the squares of a head: PER elements in each of LANES lanes (a power of two).  Adjacent elements first and in
// sixty-fourths of the head whatever LANES is, so that a row has the same sum in every kernel (fmaf by name: of a sum of two
// products either may be the one that is rounded).
template <int PER, int LANES>
__device__ __forceinline__ float sum_of_squares(const float (&v)[PER]) {
  constexpr int kEach = PER * LANES / 64, kParts = PER / kEach;
  float part[kParts];
#pragma unroll
  for (int i = 0; i < kParts; ++i) {
    part[i] = 0.f;
#pragma unroll
    for (int e = 0; e < kEach; ++e) part[i] = fmaf(v[i * kEach + e], v[i * kEach + e], part[i]);
  }
#pragma unroll
  for (int n = kParts / 2; n >= 1; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i) part[i] = part[2 * i] + part[2 * i + 1];
  return sum_over_lanes<LANES>(part[0]);
}

// Gate of a value head: a + dt_bias and the softplus live in the promoted dtype of the two operands.
__device__ __forceinline__ float decay_of(float a, float a_log, float bias, int sum_dt) {
  const float apb = round_through(a + bias, sum_dt);
  const float sp = round_through(fmaxf(apb, 0.f) + log1pf(expf(-fabsf(apb))), sum_dt);
  return expf(-expf(a_log) * sp);
}

constexpr int kTaps = 4, kKeep = kTaps - 1;

struct BlockArgs {
  const uint16_t* qkv;         // [slots, T, C], rows and slots with a stride (elements)
  const uint16_t* conv_state;  // [slots, 3, C] or null (zeros)
  const uint16_t* conv_w;      // [C, 4]
  const uint16_t *a, *b;       // [slots, T, Hv], likewise with strides
  const void *A_log, *dt_bias;  // [Hv]
  uint16_t *conv_next, *k_out, *qkv_out;  // [slots, 3, C]; [slots, T, Hk, D] and [slots, T, C] or null
  float* g_out;                           // [slots, T, Hv] or null
  long long qkv_slot, qkv_row, a_slot, a_row, b_slot, b_row;
  int param_dt;
  float eps, scale_q, scale_k;  // scales already rounded to bf16
};

// v rounded to bf16, two elements to a conversion.
template <int PER>
__device__ __forceinline__ void round_to_bf16(float (&v)[PER]) {
  typedef __attribute__((ext_vector_type(2))) __bf16 pair_t;
  typedef __attribute__((ext_vector_type(2))) float floats_t;
#pragma unroll
  for (int e = 0; e + 1 < PER; e += 2) {
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector((floats_t{v[e], v[e + 1]}), pair_t));
    v[e] = __uint_as_float(w << 16), v[e + 1] = __uint_as_float(w & 0xffff0000u);
  }
  if constexpr (PER % 2 != 0) v[PER - 1] = round_through(v[PER - 1], DFLASH_BF16);
}

// The words of a bf16 load, stored as they are.
template <int PER>
__device__ __forceinline__ void store_words(uint16_t* dst, const uint32_t (&raw)[PER]) {
  if constexpr (PER % 4 == 0) {
#pragma unroll
    for (int e = 0; e < PER; e += 4) *reinterpret_cast<uint2*>(dst + e) = uint2{raw[e / 2], raw[e / 2 + 1]};
  } else if constexpr (PER == 2) {
    *reinterpret_cast<uint32_t*>(dst) = raw[0];
  } else {
    *dst = (uint16_t)raw[0];
  }
}

// bf16 numbers held as floats, stored.
template <int PER>
__device__ __forceinline__ void store_exact(uint16_t* dst, const float (&v)[PER]) {
  uint32_t words[PER] = {};
#pragma unroll
  for (int e = 0; e + 1 < PER; e += 2) words[e / 2] = __builtin_amdgcn_perm(__float_as_uint(v[e + 1]), __float_as_uint(v[e]), 0x07060302u);
  if constexpr (PER == 1) words[0] = __float_as_uint(v[0]) >> 16;
  store_words<PER>(dst, words);
}

// PER adjacent channels (from c on) at STEPS steps from t on: rows t .. t + STEPS + 2 of [conv_state | qkv] and the taps, as loaded.
template <int PER, int STEPS = 1>
struct ConvRows {
  uint32_t x[kKeep + STEPS][PER], w[PER * kTaps];
};
// Every load is unconditional: a row that does not count (no conv state, steps past the block) is some readable row.
template <int PER, int STEPS>
__device__ __forceinline__ void request_rows(const BlockArgs& p, int slot, int t, int T, int C, int c, ConvRows<PER, STEPS>& r) {
  const uint16_t* const qkv = p.qkv + (size_t)slot * p.qkv_slot;
  const uint16_t* const before = p.conv_state + (size_t)slot * kKeep * C;
  const uint32_t pitch = (uint32_t)p.qkv_row;  // (16 rows of it are within 32 bits: checked where the launch is)
#pragma unroll
  for (int j = 0; j < kKeep + STEPS; ++j) {
    const int row = t + j, s = row - kKeep < T ? row - kKeep : T - 1;
    if (j >= kKeep) {
      load_adjacent_raw<PER>(qkv, (uint32_t)s * pitch + (uint32_t)c, false, r.x[j]);
    } else {
      const bool stored = row < kKeep && p.conv_state != nullptr;
      load_adjacent_raw<PER>(stored ? before : qkv, (stored ? (uint32_t)row * (uint32_t)C : (uint32_t)(s < 0 ? 0 : s) * pitch) + (uint32_t)c, false,
                             r.x[j]);
    }
  }
  load_adjacent_raw<PER * kTaps>(p.conv_w, (size_t)c * kTaps, false, r.w);
}

// silu(conv), and what the rows leave behind where `keeps`: the next conv state and qkv in one piece.
template <int PER, int STEPS>
__device__ __forceinline__ void convolve(const BlockArgs& p, int slot, int t, int T, int C, int c, bool keeps, ConvRows<PER, STEPS>& r,
                                         float (&act)[STEPS][PER]) {
  if (p.conv_state == nullptr) {
#pragma unroll
    for (int j = 0; j < kKeep; ++j)
#pragma unroll
      for (int e = 0; e < PER; ++e) r.x[j][e] = t + j >= kKeep ? r.x[j][e] : 0u;
  }
  float x[kKeep + STEPS][PER], w[PER * kTaps];
#pragma unroll
  for (int j = 0; j < kKeep + STEPS; ++j) unpack_adjacent<PER>(r.x[j], DFLASH_BF16, x[j]);
  unpack_adjacent<PER * kTaps>(r.w, DFLASH_BF16, w);
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    float sig[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < kTaps; ++j) acc += x[i + j][e] * w[e * kTaps + j];
      act[i][e] = acc;
    }
    round_to_bf16(act[i]);
#pragma unroll
    for (int e = 0; e < PER; ++e) sig[e] = sigmoid_of_half(act[i][e]);
    round_to_bf16(sig);
#pragma unroll
    for (int e = 0; e < PER; ++e) act[i][e] *= sig[e];
    round_to_bf16(act[i]);
  }
  if (!keeps) return;
  uint16_t* const next = p.conv_next + (size_t)slot * kKeep * C + c;
  if (t == 0) {  // blocks shorter than the state: old rows move up
#pragma unroll
    for (int row = 1; row < kKeep; ++row)
      if (row >= T) store_words<PER>(next + (size_t)(row - T) * C, r.x[row]);
  }
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    if (t + i >= T) return;
    if (t + i + kKeep >= T) store_words<PER>(next + (size_t)(t + i + kKeep - T) * C, r.x[i + kKeep]);
    if (p.qkv_out != nullptr) store_words<PER>(p.qkv_out + ((size_t)slot * T + t + i) * C + c, r.x[i + kKeep]);
  }
}

// q or k of the head from its activation: scale * rms_norm, rounded as the array it would be stored in.
template <int PER>
__device__ __forceinline__ void scale_rounded(float (&v)[PER], float inv_rms, float scale) {
#pragma unroll
  for (int e = 0; e < PER; ++e) v[e] *= inv_rms;
  round_to_bf16(v);
#pragma unroll
  for (int e = 0; e < PER; ++e) v[e] *= scale;
  round_to_bf16(v);
}
template <int PER, int LANES>
__device__ __forceinline__ void normalise(float (&v)[PER], float scale, float eps) {
  scale_rounded(v, 1.0f / sqrtf(sum_of_squares<PER, LANES>(v) / (float)(PER * LANES) + eps), scale);
}
// 1 / rms of one row, and of two: there the even lanes have the root and the quotient of the first, the odd ones those of the second.
template <int PER, int LANES>
__device__ __forceinline__ void inv_rms_of(const float (&v)[1][PER], float eps, float (&inv_rms)[1]) {
  inv_rms[0] = 1.0f / sqrtf(sum_of_squares<PER, LANES>(v[0]) / (float)(PER * LANES) + eps);
}
template <int PER, int LANES>
__device__ __forceinline__ void inv_rms_of(const float (&v)[2][PER], float eps, float (&inv_rms)[2]) {
  const float first = sum_of_squares<PER, LANES>(v[0]), second = sum_of_squares<PER, LANES>(v[1]);
  const float mine = 1.0f / sqrtf((threadIdx.x & 1 ? second : first) / (float)(PER * LANES) + eps);
  inv_rms[0] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mine), 0xA0, 0xF, 0xF, true));  // quad_perm [0,0,2,2]
  inv_rms[1] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mine), 0xF5, 0xF, 0xF, true));  // quad_perm [1,1,3,3]
}
template <int PER, int LANES>
__device__ __forceinline__ void normalise(float (&v)[2][PER], float scale, float eps) {
  float inv_rms[2];
  inv_rms_of<PER, LANES>(v, eps, inv_rms);
  scale_rounded(v[0], inv_rms[0], scale);
  scale_rounded(v[1], inv_rms[1], scale);
}

// The gate and beta of step t of value head hv, as loaded and as the recurrence reads them.
struct GateBits {
  uint32_t a, b, a_log, bias;
};
__device__ __forceinline__ GateBits request_gates(const BlockArgs& p, int slot, int t, int hv) {
  const bool wide = p.param_dt == DFLASH_FP32;
  return {p.a[(size_t)slot * p.a_slot + (size_t)t * p.a_row + hv], p.b[(size_t)slot * p.b_slot + (size_t)t * p.b_row + hv],
          load_one(p.A_log, hv, wide), load_one(p.dt_bias, hv, wide)};
}
__device__ __forceinline__ float gate_of(const BlockArgs& p, const GateBits& r) {
  return decay_of(bits_as_f32(r.a, DFLASH_BF16), bits_as_f32(r.a_log, p.param_dt), bits_as_f32(r.bias, p.param_dt),
                  p.param_dt == DFLASH_FP32 ? DFLASH_FP32 : DFLASH_BF16);
}
__device__ __forceinline__ float beta_of(const GateBits& r) {
  return round_through(sigmoid_for(bits_as_f32(r.b, DFLASH_BF16), DFLASH_BF16), DFLASH_BF16);
}

}  // namespace
}  // namespace dflash
