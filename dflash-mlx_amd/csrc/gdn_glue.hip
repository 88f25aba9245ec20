// GatedDeltaNet layer glue for gfx950: everything between the input projections and the
// recurrence in one launch, and the gated output norm in another.
//
// Mirrors the array operators of the reference's speculative GDN call
// (dflash_mlx/runtime.py:381-407 and :448): mask, depthwise causal conv over
// [conv_state | qkv], silu, split into q / k / v heads, rms_norm and scaling of q and k,
// g = exp(-exp(A_log) * softplus(a + dt_bias)), beta = sigmoid(b), the next conv state;
// then rms_norm(out, weight) * silu(z).  Every array-level operator of that sequence rounds
// to the array dtype once; the arithmetic inside an operator is fp32.
//
// For a verify block these operators are a few hundred KB per layer, and the point of fusing them is the launch
// count (two launches instead of about twenty elementwise kernels; none of their own where gdn_forward.hip takes the
// projections as they are).  For a prompt they are bound by the vector
// instructions per element (the sigmoid's exponential and division, the roundings): a wave takes several tokens
// of its head in turn, so that a row of qkv is read and unpacked once and not once per tap, the taps once per wave, and
// the gates of all its tokens are computed side by side, one token per lane.  1024 tokens of 16 + 16 + 32 heads of
// 128: 62 us with a wave per token and head, 21.4 us with several tokens, 18.6 us with rows asked for two tokens ahead, 16.2 us with
// the sigmoid of 16-bit numbers in half the instructions (glue_device.h; 4096 tokens 56.0 -> 46.7); the gated norm 15 -> 10.1 ->
// 8.4 -> 7.3 us.  With two roundings to a conversion and two tokens that share a root and a quotient (a sixth of the vector instructions gone; 128
// registers), measured back to back: 300 tokens 7.9 -> 7.3, 600 12.7 -> 10.9, 1024 17.2 -> 15.0, 2048 27.8 -> 23.0; the gated norm of 200, 1024
// and 2048 tokens of 32 heads 3.6 -> 3.2, 7.2 -> 6.5, 12.8 -> 12.5 (64 heads, 2048 tokens: 22.6 -> 19.9).  The projections are read where a joint product
// left them (rows with a stride), which saves four copies per layer call (25 us of the same prompt, 12 us of a
// verify block).
#include "gdn_block_device.h"

#include <cmath>
#include <type_traits>

namespace dflash {
namespace {

constexpr int kWavesPerGroup = 4;
constexpr int kMaxPerLane = 4;  // head dims up to 256

struct PrepareArgs {
  const void* qkv;         // [B, S, C], rows and batches with a stride
  const void* conv_state;  // [B, K-1, C] or null (zeros)
  const void* conv_w;      // [C, K]
  const void* a;           // [B, S, Hv], likewise
  const void* b;           // [B, S, Hv], likewise
  const void* A_log;       // [Hv]
  const void* dt_bias;     // [Hv]
  const uint8_t* mask;     // [B, S] or null
  void* conv_next;         // [B, K-1, C]
  void* q;                 // [B, S, Hk, Dk]
  void* k;                 // [B, S, Hk, Dk]
  void* v;                 // [B, S, Hv, Dv]
  float* g;                // [B, S, Hv]
  void* beta;              // [B, S, Hv]
  void* qkv_out;           // [B, S, C]: qkv with masked rows zeroed, or null
  long long qkv_batch, qkv_row, a_batch, a_row, b_batch, b_row;  // strides, elements
  int tokens;              // per wave
  Divisor heads, runs;     // by the waves of a run of tokens, by the runs of a batch element
  int B, S, Hk, Hv, Dk, Dv, param_dt;
  float eps, scale_q, scale_k;  // scales already rounded to the array dtype
};

// Products of fp32 numbers, before they are rounded to fp16: the compiler makes one instruction, with one rounding, of
// some products and their conversion and not of others, and a row has the same bits wherever it is computed.
template <int DT, int PER>
__device__ __forceinline__ float (&whole(float (&v)[PER]))[PER] {
  if constexpr (DT == DFLASH_FP16) {
#pragma unroll
    for (int e = 0; e < PER; ++e) asm("" : "+v"(v[e]));
  }
  return v;
}
// v rounded to the array dtype
template <int DT, int PER>
__device__ __forceinline__ void rounded(float (&v)[PER]) {
  if constexpr (DT == DFLASH_BF16) {
    round_to_bf16(v);
  } else {
    whole<DT>(v);
#pragma unroll
    for (int e = 0; e < PER; ++e) v[e] = round_through(v[e], DT);
  }
}

// LANES lanes per (batch, run of tokens, head); heads 0..Hk-1 are q, Hk..2Hk-1 are k, the rest v, those of a wave of
// one kind.  A lane holds PER = D / LANES adjacent channels of its head, so a row of the head is one access per lane
// and the K taps of those channels are PER * K adjacent weights.  All loads the first token needs are issued
// before anything is computed, and the row of the token after the next while one is worked on.
template <int DT, int PER, int K, int LANES>
__device__ __forceinline__ void prepare_head(const PrepareArgs& p, int b, int s0, int s1, bool is_v, int h, int lane) {
  const int key_dim = p.Hk * p.Dk;
  const int C = 2 * key_dim + p.Hv * p.Dv;
  constexpr int keep = K - 1;
  constexpr bool wide = DT == DFLASH_FP32;
  const int cb = is_v ? 2 * key_dim + (h - 2 * p.Hk) * p.Dv : h * p.Dk;  // q and k heads are contiguous
  const int c = cb + PER * lane;
  const int hv = is_v ? h - 2 * p.Hk : 0;
  const bool pwide = p.param_dt == DFLASH_FP32;
  const size_t qkv0 = (size_t)b * p.qkv_batch + c, token0 = (size_t)b * p.S;
  // the mask byte of a row of qkv; without a mask some byte that is not looked at
  auto mask_at = [&](int s) __attribute__((always_inline)) -> uint32_t {
    return *(p.mask != nullptr ? p.mask + token0 + s : (const uint8_t*)p.qkv);
  };
  // Every load below is unconditional: which row of which array a tap comes from, and whether it
  // counts at all, is decided by selecting the address (a tap that does not count reads some
  // readable row and is zeroed afterwards).  Loads inside branches, with the registers they
  // write preset to zero, make the compiler wait for earlier loads that used the same registers.
  uint32_t xr[K][PER], wr[PER * K], mask_byte[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const int r = s0 + j;  // row of [conv_state | qkv]
    const bool from_state = r < keep, stored = from_state && p.conv_state != nullptr;
    const int s = from_state ? 0 : r - keep;
    load_adjacent_raw<PER>(stored ? p.conv_state : p.qkv,
                           stored ? ((size_t)b * keep + r) * C + c : qkv0 + (size_t)s * p.qkv_row, wide, xr[j]);
    mask_byte[j] = mask_at(s);
  }
  uint32_t ahead[PER], mask_ahead;  // of the second token
  {
    const int s = s0 + 1 < s1 ? s0 + 1 : s0;
    load_adjacent_raw<PER>(p.qkv, qkv0 + (size_t)s * p.qkv_row, wide, ahead);
    mask_ahead = mask_at(s);
  }
  load_adjacent_raw<PER * K>(p.conv_w, (size_t)c * K, wide, wr);
  // gates of the value head's tokens, one per lane (key heads read some and do not use them)
  const int gate_token = s0 + lane < s1 ? s0 + lane : s1 - 1;
  const uint32_t a_bits = load_one(p.a, (size_t)b * p.a_batch + (size_t)gate_token * p.a_row + hv, wide);
  const uint32_t b_bits = load_one(p.b, (size_t)b * p.b_batch + (size_t)gate_token * p.b_row + hv, wide);
  const uint32_t a_log_bits = load_one(p.A_log, hv, pwide);
  const uint32_t bias_bits = load_one(p.dt_bias, hv, pwide);
  asm volatile("" ::: "memory");  // every request above is out before the first value is interpreted
  float x[K + 1][PER], w[PER * K];
#pragma unroll
  for (int j = 0; j < keep; ++j) {
    const bool from_state = s0 + j < keep;
    const bool on = from_state ? p.conv_state != nullptr : p.mask == nullptr || mask_byte[j] != 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) xr[j][e] = on ? xr[j][e] : 0u;
    unpack_adjacent<PER>(xr[j], DT, x[j]);
  }
  unpack_adjacent<PER * K>(wr, DT, w);
  if (is_v && lane < s1 - s0) {
    const float gate_a = bits_as_f32(a_bits, DT), gate_b = bits_as_f32(b_bits, DT);
    const float a_log = bits_as_f32(a_log_bits, p.param_dt), bias = bits_as_f32(bias_bits, p.param_dt);
    const size_t at = (token0 + gate_token) * p.Hv + hv;
    p.g[at] = decay_of(gate_a, a_log, bias, pwide ? DFLASH_FP32 : DT);
    store_from_f32(p.beta, at, sigmoid_for(gate_b, DT), DT);
  }
  if (s0 == 0) {
    for (int r = p.S; r < keep; ++r) {  // blocks shorter than the state: old rows move up
      float old[PER];
#pragma unroll
      for (int e = 0; e < PER; ++e) old[e] = 0.f;
      if (p.conv_state) load_adjacent<PER>(p.conv_state, ((size_t)b * keep + r) * C + c, DT, old);
      store_adjacent<PER>(p.conv_next, ((size_t)b * keep + (r - p.S)) * C + c, DT, old);
    }
  }

  auto request = [&](int s, uint32_t (&row)[PER], uint32_t& mask_of_row) __attribute__((always_inline)) {
    if (s >= s1) return;
    load_adjacent_raw<PER>(p.qkv, qkv0 + (size_t)s * p.qkv_row, wide, row);
    mask_of_row = mask_at(s);
  };
  auto bring = [&](float (&to)[PER], const uint32_t (&row)[PER], uint32_t mask_of_row) __attribute__((always_inline)) {
    const bool on = p.mask == nullptr || mask_of_row != 0;
    uint32_t words[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) words[e] = on ? row[e] : 0u;
    unpack_adjacent<PER>(words, DT, to);
  };
  // One token, or two that share a root
  auto tokens = [&](int s, auto many, uint32_t (&row)[PER], uint32_t& mask_of_row) __attribute__((always_inline)) {
    constexpr int N = decltype(many)::value;
    bring(x[keep], row, mask_of_row);
    if constexpr (N == 2) bring(x[keep + 1], ahead, mask_ahead);
    request(s + 2, row, mask_of_row);
    if constexpr (N == 2) request(s + 3, ahead, mask_ahead);
    float act[N][PER];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      // the last `keep` rows of [conv_state | qkv] are the next conv state
      if (s + i + keep >= p.S) store_adjacent<PER>(p.conv_next, ((size_t)b * keep + (s + i + keep - p.S)) * C + c, DT, x[keep + i]);
      if (p.qkv_out != nullptr) store_adjacent<PER>(p.qkv_out, (token0 + s + i) * C + c, DT, x[keep + i]);
      float sig[PER];
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < K; ++j) acc += x[i + j][e] * w[e * K + j];
        act[i][e] = acc;
      }
      rounded<DT>(act[i]);
#pragma unroll
      for (int e = 0; e < PER; ++e) sig[e] = sigmoid_for(act[i][e], DT);
      rounded<DT>(sig);
#pragma unroll
      for (int e = 0; e < PER; ++e) act[i][e] *= sig[e];
    }
#pragma unroll
    for (int j = 0; j < keep; ++j)
#pragma unroll
      for (int e = 0; e < PER; ++e) x[j][e] = x[j + N][e];
    if (is_v) {
#pragma unroll
      for (int i = 0; i < N; ++i) store_adjacent<PER>(p.v, ((token0 + s + i) * p.Hv + hv) * p.Dv + PER * lane, DT, whole<DT>(act[i]));
      return;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) rounded<DT>(act[i]);
    float inv_rms[N];
    inv_rms_of<PER, LANES>(act, p.eps, inv_rms);
    const bool is_q = h < p.Hk;
    const float scale = is_q ? p.scale_q : p.scale_k;
    void* out = is_q ? p.q : p.k;
#pragma unroll
    for (int i = 0; i < N; ++i) {
#pragma unroll
      for (int e = 0; e < PER; ++e) act[i][e] *= inv_rms[i];
      rounded<DT>(act[i]);
#pragma unroll
      for (int e = 0; e < PER; ++e) act[i][e] *= scale;
      store_adjacent<PER>(out, ((token0 + s + i) * p.Hk + (is_q ? h : h - p.Hk)) * p.Dk + PER * lane, DT, whole<DT>(act[i]));
    }
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  int s = s0;
  if constexpr (PER == 8) {
#pragma unroll 1
    for (; s + 1 < s1; s += 2) tokens(s, Two{}, xr[keep], mask_byte[keep]);
    if (s < s1) tokens(s, One{}, xr[keep], mask_byte[keep]);
  } else {  // (a wave has one token or a few, and the longer way through a second form of the code costs more than a root: 100 tokens in fp32 8.0 -> 10.3 us)
#pragma unroll 1
    for (; s < s1; s += 2) {
      tokens(s, One{}, xr[keep], mask_byte[keep]);
      if (s + 1 < s1) tokens(s + 1, One{}, ahead, mask_ahead);
    }
  }
}

template <int DT, int K>
__global__ __launch_bounds__(kWavesPerGroup * 64) void gdn_prepare_kernel(PrepareArgs p) {
  const int lane = threadIdx.x & 63;
  const int heads = (int)p.heads.by, runs = (int)p.runs.by;
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6)));
  if (w >= p.B * runs * heads) return;
  const int run = p.heads.quotient(w), h = w - run * heads;
  const int b = p.runs.quotient(run), s0 = (run - b * runs) * p.tokens;
  const int s1 = s0 + p.tokens < p.S ? s0 + p.tokens : p.S;
  const bool is_v = h >= 2 * p.Hk;
  switch ((is_v ? p.Dv : p.Dk) / 64) {
    case 1: prepare_head<DT, 1, K, 64>(p, b, s0, s1, is_v, h, lane); break;
    case 2: prepare_head<DT, 2, K, 64>(p, b, s0, s1, is_v, h, lane); break;
    case 3: prepare_head<DT, 3, K, 64>(p, b, s0, s1, is_v, h, lane); break;
    default: prepare_head<DT, 4, K, 64>(p, b, s0, s1, is_v, h, lane); break;
  }
}
// Eight channels per lane, several heads per wave: Dk = Dv = 64, 128 or 256, the q and k heads together and the v heads multiples of those
// of a wave, 16-bit arrays.  Four waves per SIMD, as the launch assumes: 130 registers without the bound, 128 and no spills with it.
template <int DT, int K, int LANES>
__global__ __launch_bounds__(kWavesPerGroup * 64) __attribute__((amdgpu_waves_per_eu(4, 4))) void gdn_prepare_wide_kernel(PrepareArgs p) {
  constexpr int kHeads = 64 / LANES;
  const int lane = threadIdx.x & 63;
  const int groups = (int)p.heads.by, runs = (int)p.runs.by;
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6)));
  if (w >= p.B * runs * groups) return;
  const int run = p.heads.quotient(w), h0 = (w - run * groups) * kHeads;
  const int b = p.runs.quotient(run), s0 = (run - b * runs) * p.tokens;
  const int s1 = s0 + p.tokens < p.S ? s0 + p.tokens : p.S;
  prepare_head<DT, 8, K, LANES>(p, b, s0, s1, h0 >= 2 * p.Hk, h0 + lane / LANES, lane % LANES);
}
template <int DT>
const void* prepare_kernel_for(int conv_kernel) {
  return conv_kernel == 4   ? (const void*)gdn_prepare_kernel<DT, 4>
         : conv_kernel == 3 ? (const void*)gdn_prepare_kernel<DT, 3>
                            : (const void*)gdn_prepare_kernel<DT, 2>;
}
template <int DT, int K>
const void* wide_kernel_for(int D) {
  return D == 64    ? (const void*)gdn_prepare_wide_kernel<DT, K, 8>
         : D == 128 ? (const void*)gdn_prepare_wide_kernel<DT, K, 16>
                    : (const void*)gdn_prepare_wide_kernel<DT, K, 32>;
}
template <int DT>
const void* wide_kernel_for(int D, int conv_kernel) {
  return conv_kernel == 4 ? wide_kernel_for<DT, 4>(D) : conv_kernel == 3 ? wide_kernel_for<DT, 3>(D) : wide_kernel_for<DT, 2>(D);
}

struct NormArgs {
  const void* x;       // [B, T, H, D]
  const void* z;       // [B, T, H, D], tokens and batches with a stride
  const void* weight;  // [D]
  void* y;             // like x
  long long z_batch, z_row;
  int rows, T, H;      // rows = B T H
  Divisor heads, tokens;  // by H, by T
  int per_wave;        // rows of a wave
  int D, weight_dt;
  float eps;
};

// LANES lanes for a few rows, `step` apart: rms_norm(x, weight) * silu(z); a lane holds PER = D / LANES adjacent elements.
template <int DT, int PER, int LANES>
__device__ __forceinline__ void gated_norm_rows(const NormArgs& p, int row, int end, int step, int lane) {
  constexpr bool wide = DT == DFLASH_FP32;
  auto rounded = [](float (&v)[PER]) __attribute__((always_inline)) {
    if constexpr (DT == DFLASH_BF16) {
      round_to_bf16(v);
    } else {
#pragma unroll
      for (int e = 0; e < PER; ++e) v[e] = round_through(v[e], DT);
    }
  };
  uint32_t xr[2][PER], zr[2][PER], wr[PER];
  auto load = [&](int i, int r) __attribute__((always_inline)) {
    const int token = p.heads.quotient(r), h = r - token * p.H, b = p.tokens.quotient(token), t = token - b * p.T;
    load_adjacent_raw<PER>(p.x, (size_t)r * p.D + PER * lane, wide, xr[i]);
    load_adjacent_raw<PER>(p.z, (size_t)b * p.z_batch + (size_t)t * p.z_row + (size_t)h * p.D + PER * lane, wide, zr[i]);
  };
  load(0, row < end ? row : end - 1);
  load_adjacent_raw<PER>(p.weight, PER * lane, p.weight_dt == DFLASH_FP32, wr);
  if (row + step < end) load(1, row + step);
  asm volatile("" ::: "memory");  // all requests are out before the first value is interpreted
  float wt[PER];
  unpack_adjacent<PER>(wr, p.weight_dt, wt);
  // one row, or two that share a root
  auto rows = [&](auto many) __attribute__((always_inline)) {
    constexpr int N = decltype(many)::value;
    float x[N][PER], z[N][PER], inv_rms[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      unpack_adjacent<PER>(xr[i], DT, x[i]);
      unpack_adjacent<PER>(zr[i], DT, z[i]);
    }
    if constexpr (N == 2) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (row + (2 + i) * step < end) load(i, row + (2 + i) * step);
    }
    inv_rms_of<PER, LANES>(x, p.eps, inv_rms);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float y[PER];
#pragma unroll
      for (int e = 0; e < PER; ++e) y[e] = sigmoid_for(z[i][e], DT);
      rounded(y);
#pragma unroll
      for (int e = 0; e < PER; ++e) y[e] *= z[i][e];
      rounded(y);
#pragma unroll
      for (int e = 0; e < PER; ++e) x[i][e] = x[i][e] * inv_rms[i] * wt[e];
      rounded(x[i]);
#pragma unroll
      for (int e = 0; e < PER; ++e) y[e] *= x[i][e];
      store_adjacent<PER>(p.y, (size_t)row * p.D + (size_t)i * step * p.D + PER * lane, DT, y);
    }
  };
#pragma unroll 1
  for (; row + step < end; row += 2 * step) rows(std::integral_constant<int, 2>{});
  if (row < end) rows(std::integral_constant<int, 1>{});
}

template <int DT>
__global__ __launch_bounds__(kWavesPerGroup * 64) void gdn_gated_norm_kernel(NormArgs p) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6)));
  const long long first = (long long)w * p.per_wave;
  if (first >= p.rows) return;
  const int row = (int)first, end = p.rows - row < p.per_wave ? p.rows : row + p.per_wave;
  switch (p.D / 64) {
    case 1: gated_norm_rows<DT, 1, 64>(p, row, end, 1, lane); break;
    case 2: gated_norm_rows<DT, 2, 64>(p, row, end, 1, lane); break;
    case 3: gated_norm_rows<DT, 3, 64>(p, row, end, 1, lane); break;
    default: gated_norm_rows<DT, 4, 64>(p, row, end, 1, lane); break;
  }
}

template <int DT, int LANES>
__global__ __launch_bounds__(kWavesPerGroup * 64) void gdn_gated_norm_wide_kernel(NormArgs p) {
  constexpr int kRows = 64 / LANES;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6)));
  const long long first = (long long)w * p.per_wave;
  if (first >= p.rows) return;
  const int row = (int)first, end = p.rows - row < p.per_wave ? p.rows : row + p.per_wave;
  gated_norm_rows<DT, 8, LANES>(p, row + lane / LANES, end, kRows, lane % LANES);
}
template <int DT>
const void* wide_norm_for(int D) {
  return D == 64    ? (const void*)gdn_gated_norm_wide_kernel<DT, 8>
         : D == 128 ? (const void*)gdn_gated_norm_wide_kernel<DT, 16>
                    : (const void*)gdn_gated_norm_wide_kernel<DT, 32>;
}

bool known_dtype(int dt) { return dt == DFLASH_BF16 || dt == DFLASH_FP16 || dt == DFLASH_FP32; }
bool head_dim_ok(int d) { return d > 0 && d % 64 == 0 && d <= 64 * kMaxPerLane; }

// the value a Python float takes when it meets an array of dtype dt
float as_array_scalar(double v, int dt) {
  const float f = (float)v;
  if (dt == DFLASH_FP32) return f;
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if (dt == DFLASH_BF16) {
    u += 0x7fffu + ((u >> 16) & 1u);
    u &= 0xffff0000u;
    float r;
    __builtin_memcpy(&r, &u, 4);
    return r;
  }
  return (float)(_Float16)f;
}

}  // namespace
}  // namespace dflash

extern "C" int dflash_gdn_prepare_rows(const void* qkv, const void* conv_state, const void* conv_w, const void* a,
                                       const void* b, const void* A_log, const void* dt_bias, const uint8_t* mask,
                                       void* conv_next, void* q, void* k, void* v, float* g, void* beta, void* qkv_out,
                                       const long long* strides, int B, int S, int Hk, int Hv, int Dk, int Dv,
                                       int conv_kernel, int dtype, int param_dtype, float eps, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(qkv && conv_w && a && b && A_log && dt_bias && conv_next && q && k && v && g && beta && strides,
                 DFLASH_ERR_ARG, "dflash_gdn_prepare: null operand");
  DFLASH_REQUIRE(known_dtype(dtype) && known_dtype(param_dtype), DFLASH_ERR_ARG,
                 "dflash_gdn_prepare: unknown dtype code");
  DFLASH_REQUIRE(B >= 0 && S >= 0 && Hk > 0 && Hv > 0 && conv_kernel >= 2 && conv_kernel <= 4, DFLASH_ERR_SHAPE,
                 "dflash_gdn_prepare: bad dimension (conv kernels of 2 to 4 taps)");
  DFLASH_REQUIRE(head_dim_ok(Dk) && head_dim_ok(Dv), DFLASH_ERR_SHAPE,
                 "dflash_gdn_prepare: head dims must be multiples of 64 up to 256, got %d and %d", Dk, Dv);
  const int heads = 2 * Hk + Hv;
  DFLASH_REQUIRE((long long)B * S * heads < (1ll << 31), DFLASH_ERR_SHAPE, "dflash_gdn_prepare: too many rows");
  if (B == 0) return DFLASH_OK;
  DFLASH_REQUIRE(S > 0, DFLASH_ERR_SHAPE, "dflash_gdn_prepare: empty block");
  for (int i = 0; i < 6; ++i) DFLASH_REQUIRE(strides[i] >= 0, DFLASH_ERR_SHAPE, "dflash_gdn_prepare: negative stride");
  PrepareArgs p;
  p.qkv = qkv; p.conv_state = conv_state; p.conv_w = conv_w; p.a = a; p.b = b; p.A_log = A_log;
  p.dt_bias = dt_bias; p.mask = mask; p.conv_next = conv_next; p.q = q; p.k = k; p.v = v; p.g = g;
  p.beta = beta; p.qkv_out = qkv_out; p.B = B; p.S = S; p.Hk = Hk; p.Hv = Hv; p.Dk = Dk; p.Dv = Dv;
  p.qkv_batch = strides[0]; p.qkv_row = strides[1]; p.a_batch = strides[2]; p.a_row = strides[3];
  p.b_batch = strides[4]; p.b_row = strides[5];
  p.param_dt = param_dtype; p.eps = eps;
  const double inv_scale = 1.0 / sqrt((double)Dk);
  p.scale_q = as_array_scalar(inv_scale * inv_scale, dtype);
  p.scale_k = as_array_scalar(inv_scale, dtype);
  // as many tokens per wave as leave 8 waves per SIMD: below that a wave's latency counts, not its instructions
  const long long per = (long long)B * S * heads / 8192;
  p.tokens = per < 1 ? 1 : per > 16 ? 16 : (int)per;
  // Eight channels per lane: the sums, roots and addresses of a row are then paid for four heads of 128 at a time.  From 640 such
  // waves on (16 + 16 + 32 heads of 128, us, a head and several per wave: 32 tokens 4.6 / 4.8, 40 tokens 5.3 / 4.7, 128 tokens
  // 9.7 / 5.4, 200 tokens 13.8 / 7.2, 1024 tokens 22.3 / 16.3), and as many tokens each as leave the 4 waves per SIMD that fit: a
  // few more would run by themselves at the end (3072 and 8192 waves / 4096: 512 tokens 11.3 and 13.0 / 11.2, 1024 tokens 17.8 and
  // 17.1 / 16.3).  A wave may have heads of q and of k: 4 + 4 + 8 heads of 64, a head per wave and eight, 320 tokens 5.9 / 3.7, 1024 tokens
  // 8.5 / 4.5; 2 + 2 + 8 heads of 128, 700 tokens 9.0 / 5.6.  Its accesses are of 8 bytes.
  const int per_wave = 512 / Dk;  // heads
  const uintptr_t places = (uintptr_t)qkv | (uintptr_t)conv_state | (uintptr_t)conv_w | (uintptr_t)conv_next | (uintptr_t)q | (uintptr_t)k |
                           (uintptr_t)v | (uintptr_t)qkv_out | (uintptr_t)(2 * (strides[0] | strides[1]));
  const bool wide = dtype != DFLASH_FP32 && Dk == Dv && Dk != 192 && 2 * Hk % per_wave == 0 && Hv % per_wave == 0 && places % 8 == 0 &&
                    (long long)B * S * heads / per_wave >= 640;
  if (wide) {
    const long long each = ((long long)B * S * heads / per_wave + 4095) / 4096, most = Dk / 8 < 16 ? Dk / 8 : 16;
    p.tokens = (int)(each > most ? most : each);  // (a lane of the head computes a token's gates)
  }
  p.runs = Divisor::of((S + p.tokens - 1) / p.tokens);
  p.heads = Divisor::of(wide ? heads / per_wave : heads);
  const long long waves = (long long)B * p.runs.by * p.heads.by;
  const unsigned groups = (unsigned)((waves + kWavesPerGroup - 1) / kWavesPerGroup);
  const void* fn = wide ? (dtype == DFLASH_BF16 ? wide_kernel_for<DFLASH_BF16>(Dk, conv_kernel)
                                                : wide_kernel_for<DFLASH_FP16>(Dk, conv_kernel))
                   : dtype == DFLASH_BF16 ? prepare_kernel_for<DFLASH_BF16>(conv_kernel)
                   : dtype == DFLASH_FP16 ? prepare_kernel_for<DFLASH_FP16>(conv_kernel)
                                          : prepare_kernel_for<DFLASH_FP32>(conv_kernel);
  void* args[] = {&p};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3(groups), dim3(kWavesPerGroup * 64), args, 0, (hipStream_t)stream));
  return DFLASH_OK;
}

extern "C" int dflash_gdn_prepare(const void* qkv, const void* conv_state, const void* conv_w, const void* a,
                                  const void* b, const void* A_log, const void* dt_bias, const uint8_t* mask,
                                  void* conv_next, void* q, void* k, void* v, float* g, void* beta, int B,
                                  int S, int Hk, int Hv, int Dk, int Dv, int conv_kernel, int dtype,
                                  int param_dtype, float eps, void* stream) {
  const long long row = 2ll * Hk * Dk + (long long)Hv * Dv;
  const long long strides[6] = {S * row, row, (long long)S * Hv, Hv, (long long)S * Hv, Hv};
  return dflash_gdn_prepare_rows(qkv, conv_state, conv_w, a, b, A_log, dt_bias, mask, conv_next, q, k, v, g, beta, nullptr, strides,
                                 B, S, Hk, Hv, Dk, Dv, conv_kernel, dtype, param_dtype, eps, stream);
}

namespace dflash {
// x, y [B, T, H, D] contiguous, z with these strides (also called by gdn_forward.hip)
int gdn_gated_norm_launch(const void* x, const void* z, const void* weight, void* y, int B, int T, int H, int D,
                          long long z_batch, long long z_row, int dtype, int weight_dtype, float eps, hipStream_t stream) {
  NormArgs p;
  p.x = x; p.z = z; p.weight = weight; p.y = y;
  p.z_batch = z_batch; p.z_row = z_row;
  p.rows = B * T * H; p.T = T; p.H = H; p.D = D;
  p.heads = Divisor::of(H); p.tokens = Divisor::of(T);
  p.weight_dt = weight_dtype; p.eps = eps;
  p.per_wave = p.rows / 8192 < 1 ? 1 : p.rows / 8192 > 16 ? 16 : p.rows / 8192;
  // eight elements per lane and several rows per wave where that leaves 4 waves per SIMD: 12.3 -> 10.1 us (32 768 rows of 128)
  const bool wide = dtype != DFLASH_FP32 && D != 192 && p.rows / (512 / D) >= 4096;
  if (wide) {
    const int passes = p.rows / (512 / D) / 4096;
    p.per_wave = 512 / D * (passes > 8 ? 8 : passes);
  }
  const long long waves = ((long long)p.rows + p.per_wave - 1) / p.per_wave;
  const unsigned groups = (unsigned)((waves + kWavesPerGroup - 1) / kWavesPerGroup);
  const void* fn = wide ? (dtype == DFLASH_BF16 ? wide_norm_for<DFLASH_BF16>(D) : wide_norm_for<DFLASH_FP16>(D))
                   : dtype == DFLASH_BF16 ? (const void*)gdn_gated_norm_kernel<DFLASH_BF16>
                   : dtype == DFLASH_FP16 ? (const void*)gdn_gated_norm_kernel<DFLASH_FP16>
                                          : (const void*)gdn_gated_norm_kernel<DFLASH_FP32>;
  void* args[] = {&p};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3(groups), dim3(kWavesPerGroup * 64), args, 0, stream));
  return DFLASH_OK;
}
}  // namespace dflash

extern "C" int dflash_gdn_gated_norm(const void* x, const void* z, const void* weight, void* y, long long rows,
                                     int D, int dtype, int weight_dtype, float eps, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(x && z && weight && y, DFLASH_ERR_ARG, "dflash_gdn_gated_norm: null operand");
  DFLASH_REQUIRE(known_dtype(dtype) && known_dtype(weight_dtype), DFLASH_ERR_ARG,
                 "dflash_gdn_gated_norm: unknown dtype code");
  DFLASH_REQUIRE(rows >= 0 && rows < (1ll << 31), DFLASH_ERR_SHAPE, "dflash_gdn_gated_norm: bad row count");
  DFLASH_REQUIRE(head_dim_ok(D), DFLASH_ERR_SHAPE,
                 "dflash_gdn_gated_norm: row length must be a multiple of 64 up to 256, got %d", D);
  if (rows == 0) return DFLASH_OK;
  return gdn_gated_norm_launch(x, z, weight, y, 1, 1, (int)rows, D, 0, 0, dtype, weight_dtype, eps, (hipStream_t)stream);
}
