// Glue of a gated attention layer for gfx950: everything between its projections and the attention in
// one launch, and the output gate in another.
//
// Replaces the array operators of dflash_mlx/runtime.py:527-556 (split of q_proj into queries and gate, head
// norms, rotary embedding, cache update) and :606-616 (output * sigmoid(gate)).  Every operator rounds to the
// array dtype once and is fp32 inside, the rotation's products and sums one rounding each, as the array
// operators do it.
//
// What bounds it is neither bandwidth (a block of 16 tokens is about 1 MB) nor arithmetic: as array operators the
// same steps were 70 launches, 2 to 5 us each on the device and about 400 us of host time per layer call.
// Measured, 16 tokens of 32 + 8 heads of 256: layer call over 4 112 or 32 716 keys
// 498 -> 109 us (host time: the kernels are 62 and 102 us); this kernel 5.8 us, 4.5 with the angles once per workgroup (300 tokens of
// 16 + 2 heads 12.8 -> 7.8), the gate 4 us (a verify block over a
// long cache has it in the merge of sdpa_q16.hip instead).
#include "glue_device.h"

#include <cmath>

namespace dflash {
namespace {

constexpr int kWavesPerGroup = 4;

struct AttnPrepareArgs {
  const uint16_t *q, *k, *v;  // [B, L, Hq, 2 D] (queries, gate), [B, L, Hk, D] twice; heads and features contiguous
  long long q_batch, q_row, k_batch, k_row, v_batch, v_row;
  const void *q_weight, *k_weight;  // [D]
  uint16_t* q_out;                  // [B, Hq, L, D]
  uint16_t *k_out, *v_out;          // rows of a cache, [B, Hk, L, D] with these strides
  long long ko_batch, ko_head, ko_row, vo_batch, vo_head, vo_row;
  int B, L, Hq, Hk, half, offset, dt, q_weight_dt, k_weight_dt;
  int waves;  // per token; each takes every waves-th head
  Divisor groups, tokens;  // by the workgroups of a token, by L
  float q_eps, k_eps, base, inv_half;
};

// A workgroup has one token: its angles, the same for every head, are computed once, one per thread, while the first rows are on
// their way (before, each wave for itself: four powers, cosines and sines per lane of a head of 256, more than half of a wave's
// instructions).
template <int PER>
__global__ __launch_bounds__(kWavesPerGroup * 64) void attn_prepare_kernel(AttnPrepareArgs p) {
#pragma clang fp contract(off)
  constexpr int D = 64 * PER;
  __shared__ float2 turn[D / 2];  // cosine and sine
  const int rotated = p.Hq + p.Hk, heads = rotated + p.Hk;
  const int token = p.groups.quotient((int)blockIdx.x), b = p.tokens.quotient(token), l = token - b * p.L;
  const int first = ((int)blockIdx.x - token * (int)p.groups.by) * kWavesPerGroup + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = PER * lane;
  const bool rotates = c < 2 * p.half, upper = c >= p.half;
  const int other = rotates ? (upper ? lane - p.half / PER : lane + p.half / PER) : lane;
  uint32_t raw[PER], wraw[PER];
  auto request = [&](int h) __attribute__((always_inline)) {
    const int hk = h - p.Hq;
    const bool is_q = h < p.Hq, is_v = h >= rotated;
    const uint16_t* const src = is_q   ? p.q + b * p.q_batch + l * p.q_row + (size_t)h * (2 * D)
                                : is_v ? p.v + b * p.v_batch + l * p.v_row + (size_t)(h - rotated) * D
                                       : p.k + b * p.k_batch + l * p.k_row + (size_t)hk * D;
    load_adjacent_raw<PER>(src, c, false, raw);
    load_adjacent_raw<PER>(is_q ? p.q_weight : p.k_weight, c, (is_q ? p.q_weight_dt : p.k_weight_dt) == DFLASH_FP32, wraw);
  };
  const bool busy = first < p.waves && first < heads;
  if (busy) request(first);
  asm volatile("" ::: "memory");  // on their way before the angles
  if ((int)threadIdx.x < p.half) {
    const float angle = (float)(p.offset + l) * powf(p.base, -(float)(int)threadIdx.x * p.inv_half);
    turn[threadIdx.x] = make_float2(cosf(angle), sinf(angle));
  }
  __syncthreads();
  if (!busy) return;
  float cs[PER], sn[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const float2 t = turn[rotates ? (upper ? c - p.half : c) + e : 0];
    cs[e] = t.x, sn[e] = t.y;
  }
  for (int h = first; h < heads; h += p.waves) {
    if (h >= rotated) {
      uint16_t* const dst = p.v_out + b * p.vo_batch + (h - rotated) * p.vo_head + l * p.vo_row + c;
      store_raw<PER>(dst, raw);
      if (h + p.waves < heads) request(h + p.waves);
      continue;
    }
    const bool is_q = h < p.Hq;
    const int hk = h - p.Hq;
    float x[PER], w[PER];
    unpack_adjacent<PER>(raw, p.dt, x);
    unpack_adjacent<PER>(wraw, is_q ? p.q_weight_dt : p.k_weight_dt, w);
    if (h + p.waves < heads) request(h + p.waves);
    norm_and_turn<PER>(x, w, is_q ? p.q_eps : p.k_eps, cs, sn, rotates, upper, other, p.dt);
    if (is_q) {
      store_adjacent<PER>(p.q_out, (((size_t)b * p.Hq + h) * p.L + l) * D + c, p.dt, x);
    } else {
      store_adjacent<PER>(p.k_out + b * p.ko_batch + hk * p.ko_head + l * p.ko_row, c, p.dt, x);
    }
  }
}

struct AttnGateArgs {
  const uint16_t* o;     // [B, Hq, L, D], features contiguous
  const uint16_t* gate;  // [B, L, Hq, 2 D] as q_proj gives it: the gate is the second half of a head
  uint16_t* y;           // [B, L, Hq, D]
  long long o_batch, o_head, o_row, g_batch, g_row;
  long long pieces;  // of four elements
  int L, Hq, D, dt;
};

__global__ __launch_bounds__(256) void attn_gate_kernel(AttnGateArgs p) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.pieces) return;
  const int c = 4 * (int)(i % (p.D / 4));
  const long long row = i / (p.D / 4);
  const int h = (int)(row % p.Hq);
  const long long token = row / p.Hq;
  const int l = (int)(token % p.L), b = (int)(token / p.L);
  uint32_t oraw[4], graw[4];
  load_adjacent_raw<4>(p.o + b * p.o_batch + h * p.o_head + l * p.o_row, c, false, oraw);
  load_adjacent_raw<4>(p.gate + b * p.g_batch + l * p.g_row, (size_t)h * 2 * p.D + p.D + c, false, graw);
  float o[4], g[4];
  unpack_adjacent<4>(oraw, p.dt, o);
  unpack_adjacent<4>(graw, p.dt, g);
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] *= round_through(sigmoid_of_half(g[e]), p.dt);
  store_adjacent<4>(p.y, (size_t)i * 4, p.dt, o);
}

bool head_dim_ok(int d) { return d == 64 || d == 128 || d == 192 || d == 256; }
bool known_dtype(int dt) { return dt == DFLASH_BF16 || dt == DFLASH_FP16 || dt == DFLASH_FP32; }

}  // namespace
}  // namespace dflash

extern "C" int dflash_attn_prepare(const void* q, const void* k, const void* v, const void* q_weight, const void* k_weight,
                                   void* q_out, void* k_out, void* v_out, int B, int L, int Hq, int Hk, int D,
                                   int rope_dims, int offset, const long long* strides, float q_eps, float k_eps,
                                   float rope_base, int dtype, int q_weight_dtype, int k_weight_dtype, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(q && k && v && q_weight && k_weight && q_out && k_out && v_out && strides, DFLASH_ERR_ARG,
                 "dflash_attn_prepare: null operand");
  DFLASH_REQUIRE((dtype == DFLASH_BF16 || dtype == DFLASH_FP16) && known_dtype(q_weight_dtype) && known_dtype(k_weight_dtype),
                 DFLASH_ERR_ARG, "dflash_attn_prepare: activations must be bf16/fp16, norm weights bf16/fp16/fp32");
  DFLASH_REQUIRE(B > 0 && L > 0 && Hq > 0 && Hk > 0 && offset >= 0 && head_dim_ok(D), DFLASH_ERR_SHAPE,
                 "dflash_attn_prepare: B %d, L %d, Hq %d, Hk %d, offset %d, head dim %d (a multiple of 64 up to 256)", B, L, Hq,
                 Hk, offset, D);
  const int per = D / 64;
  DFLASH_REQUIRE(rope_dims > 0 && rope_dims <= D && rope_dims % (2 * per) == 0, DFLASH_ERR_SHAPE,
                 "dflash_attn_prepare: %d rotated features of %d (a multiple of %d)", rope_dims, D, 2 * per);
  uintptr_t bits = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)q_out | (uintptr_t)k_out | (uintptr_t)v_out;
  for (int i = 0; i < 12; ++i) {
    DFLASH_REQUIRE(strides[i] >= 0, DFLASH_ERR_SHAPE, "dflash_attn_prepare: negative stride");
    bits |= (uintptr_t)strides[i] * 2;
  }
  DFLASH_REQUIRE(bits % 8 == 0 && ((uintptr_t)q_weight | (uintptr_t)k_weight) % 8 == 0, DFLASH_ERR_ARG,
                 "dflash_attn_prepare: operands and rows must be 8-byte aligned");
  AttnPrepareArgs p;
  p.q = (const uint16_t*)q; p.k = (const uint16_t*)k; p.v = (const uint16_t*)v;
  p.q_batch = strides[0]; p.q_row = strides[1]; p.k_batch = strides[2]; p.k_row = strides[3];
  p.v_batch = strides[4]; p.v_row = strides[5];
  p.ko_batch = strides[6]; p.ko_head = strides[7]; p.ko_row = strides[8];
  p.vo_batch = strides[9]; p.vo_head = strides[10]; p.vo_row = strides[11];
  p.q_weight = q_weight; p.k_weight = k_weight;
  p.q_out = (uint16_t*)q_out; p.k_out = (uint16_t*)k_out; p.v_out = (uint16_t*)v_out;
  p.B = B; p.L = L; p.Hq = Hq; p.Hk = Hk; p.half = rope_dims / 2; p.offset = offset;
  p.dt = dtype; p.q_weight_dt = q_weight_dtype; p.k_weight_dt = k_weight_dtype;
  p.q_eps = q_eps; p.k_eps = k_eps; p.base = rope_base; p.inv_half = 1.0f / (float)p.half;
  // One wave per head while that leaves the chip with fewer than 8 waves per SIMD, beyond that several heads per wave.
  const long long tokens = (long long)B * L, want = (8192 + tokens - 1) / tokens;
  p.waves = want < Hq + 2 * Hk ? (int)want : Hq + 2 * Hk;
  p.groups = Divisor::of((p.waves + kWavesPerGroup - 1) / kWavesPerGroup);
  p.tokens = Divisor::of(L);
  const long long groups = tokens * p.groups.by;
  DFLASH_REQUIRE(groups * kWavesPerGroup < (1ll << 31), DFLASH_ERR_SHAPE, "dflash_attn_prepare: too many rows");
  const dim3 grid((unsigned)groups), block(kWavesPerGroup * 64);
  switch (per) {
    case 1: hipLaunchKernelGGL(attn_prepare_kernel<1>, grid, block, 0, (hipStream_t)stream, p); break;
    case 2: hipLaunchKernelGGL(attn_prepare_kernel<2>, grid, block, 0, (hipStream_t)stream, p); break;
    case 3: hipLaunchKernelGGL(attn_prepare_kernel<3>, grid, block, 0, (hipStream_t)stream, p); break;
    default: hipLaunchKernelGGL(attn_prepare_kernel<4>, grid, block, 0, (hipStream_t)stream, p); break;
  }
  DFLASH_HIP_OK(hipGetLastError());
  return DFLASH_OK;
}

extern "C" int dflash_attn_gate(const void* o, const void* gate, void* y, int B, int L, int Hq, int D, long long o_batch_stride,
                                long long o_head_stride, long long o_row_stride, long long gate_batch_stride,
                                long long gate_row_stride, int dtype, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(o && gate && y, DFLASH_ERR_ARG, "dflash_attn_gate: null operand");
  DFLASH_REQUIRE(dtype == DFLASH_BF16 || dtype == DFLASH_FP16, DFLASH_ERR_ARG, "dflash_attn_gate: bf16 or fp16 only");
  DFLASH_REQUIRE(B > 0 && L > 0 && Hq > 0 && head_dim_ok(D), DFLASH_ERR_SHAPE,
                 "dflash_attn_gate: B %d, L %d, Hq %d, head dim %d (a multiple of 64 up to 256)", B, L, Hq, D);
  const long long strides[] = {o_batch_stride, o_head_stride, o_row_stride, gate_batch_stride, gate_row_stride};
  uintptr_t bits = (uintptr_t)o | (uintptr_t)gate | (uintptr_t)y;
  for (long long s : strides) {
    DFLASH_REQUIRE(s >= 0, DFLASH_ERR_SHAPE, "dflash_attn_gate: negative stride");
    bits |= (uintptr_t)s * 2;
  }
  DFLASH_REQUIRE(bits % 8 == 0, DFLASH_ERR_ARG, "dflash_attn_gate: operands and rows must be 8-byte aligned");
  AttnGateArgs p;
  p.o = (const uint16_t*)o; p.gate = (const uint16_t*)gate; p.y = (uint16_t*)y;
  p.o_batch = o_batch_stride; p.o_head = o_head_stride; p.o_row = o_row_stride;
  p.g_batch = gate_batch_stride; p.g_row = gate_row_stride;
  p.pieces = (long long)B * L * Hq * (D / 4);
  p.L = L; p.Hq = Hq; p.D = D; p.dt = dtype;
  DFLASH_REQUIRE(p.pieces < (1ll << 38), DFLASH_ERR_SHAPE, "dflash_attn_gate: too many rows");
  hipLaunchKernelGGL(attn_gate_kernel, dim3((unsigned)((p.pieces + 255) / 256)), dim3(256), 0, (hipStream_t)stream, p);
  DFLASH_HIP_OK(hipGetLastError());
  return DFLASH_OK;
}
