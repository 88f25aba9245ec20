// Exact attention for a verify block of 16 queries over a long KV cache, gfx950.
//
// Replaces the two Metal kernels of dflash_mlx/kernels.py:442-655 (`batched_sdpa_2pass_partials`
// and `batched_sdpa_2pass_reduce`) behind `batched_sdpa_2pass_exact` (:658-761): for every
// batch b, query head hq (key/value head hk = hq / (Hq / Hk)) and query position i < 16
//     out[i] = softmax_n( scale * q[i] . k[n] + mask[i][n] ) v[n]
// over the keys n <= N - 16 + i (the block's own causal rule, kernels.py:517) whose mask value,
// if a mask is given, is not the dtype's lowest finite value (:452-454); rows without any key
// give 0 (:617).
//
// The path is bound by reading K and V once (2 * N * D * 2 bytes per key/value head; at
// N = 4096, D = 256, 8 heads: 33.7 MB per layer).  So the 16 queries of ALL query heads of a
// key/value head are served from one pass over its keys: a workgroup takes one (batch,
// key/value head, range of keys), wave w holds the 16 queries of query head hk * G + w, and
// K / V tiles of 32 keys go through LDS once for all waves.
//
// Matrix-core layout (v_mfma_f32_16x16x32 bf16 / f16; A lane l = A[l % 16][8 (l / 16) ..+7],
// B lane l = B[8 (l / 16) ..+7][l % 16], accumulator r of lane l = C[4 (l / 16) + r][l % 16]):
//   S^T = K Q^T : A = K tile rows (keys), B = Q (held in registers for the whole kernel);
//                 lane (j, kb) ends up with query j's scores for keys 4 kb + r of each
//                 16-key half: the softmax state (max, sum, rescale factor) is per lane;
//   O^T = V^T P^T: those scores, exponentiated and packed, ARE the B operand (k-slot e <-> key
//                 4 kb + e, slot 4 + e <-> key 16 + 4 kb + e), and the A operand with the same
//                 key order comes from the row-major V tile through ds_read_b64_tr_b16: within
//                 a group of 16 lanes, source lane 4 e + q supplies 8 bytes and lane t receives
//                 element t % 4 of source lanes t / 4, 4 + t / 4, 8 + t / 4, 12 + t / 4 - so source
//                 lane 4 e + q points at V[key 4 kb + e][16 c + 4 q ..+3] and lane t receives
//                 column 16 c + t of four keys.  No transposed copy of V or P is ever stored.
// Ranges of keys (splits) write partial outputs in the input dtype (kernels.py:556-558) with their
// fp32 max and sum; a second kernel merges them (the reference's second pass).
#include "glue_device.h"

#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace dflash {
namespace {

constexpr int kTileKeys = 32;
constexpr int kThreads = 512;   // eight waves
constexpr int kPadElems = 8;      // 16 bytes: rows of a tile start 16 bytes apart modulo 128
// Score of a key that is not used: below every score a used key can have (a used key may carry
// the dtype's lowest finite value as its mask, -3.39e38 for bf16).
constexpr float kMasked = -3.4028234663852886e38f;

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

struct SdpaArgs {
  const uint16_t* q;     // [B, Hq, 16, D]
  const uint16_t* k;     // [B, Hk, N, D] through strides (elements), D contiguous
  const uint16_t* v;
  const uint16_t* mask;  // [B, Hq, 16, N] additive, in the input dtype, or null
  uint16_t* out;         // [B, Hq, 16, D], gated: [B, 16, Hq, D]
  const uint16_t* gate;  // [B, 16, Hq, 2 D] with these strides (elements), the gate behind the queries of a head; or null
  long long gate_batch_stride, gate_row_stride;
  uint16_t* part_o;      // [splits, B * Hq, 16, D] in the input dtype, as the reference keeps them
  float* part_ml;        // [splits, B * Hq, 16, 2]  (max, sum)
  long long k_batch_stride, k_head_stride, k_seq_stride;
  long long v_batch_stride, v_head_stride, v_seq_stride;
  int B, Hq, Hk, N, G, splits, keys_per_split;
  Divisor ranges, key_heads, heads;  // by splits, Hk, Hq
  float scale, lowest;   // lowest finite value of the input dtype
};

// What stands between the projections and the attention of a block, where the attention's launch does it (BLOCK): queries and
// keys of the block as the projections gave them, and the cache's rows N - 16 .. N - 1, which are written here.
struct BlockArgs {
  const uint16_t *q, *k, *v;  // [B, 16, Hq, 2 D] (queries, gate), [B, 16, Hk, D] twice, through strides (elements)
  long long q_batch, q_row, k_batch, k_row, v_batch, v_row;
  const uint16_t *q_weight, *k_weight;  // [D], of the input dtype
  uint16_t *k_cache, *v_cache;          // where k and v of SdpaArgs begin
  int half;                             // rotated features / 2: 32, 64 or 128
  float q_eps, k_eps, base, inv_half;
};
template <bool BLOCK>
struct KernelArgs : SdpaArgs {};
template <>
struct KernelArgs<true> : SdpaArgs {
  BlockArgs block;
};
constexpr int kTurnPad = 2;  // pairs between the rows of the table of angles: its rows start 16 bytes apart modulo 128
constexpr size_t turn_bytes(int half) { return 16 * (size_t)(half + kTurnPad) * sizeof(float2) + half * sizeof(float); }

template <bool FP16>
__device__ __forceinline__ f32x4_t mfma32(uint4 a, uint4 b, f32x4_t c) {
  if (FP16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                  0, 0, 0);
  }
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}

template <bool FP16>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  const f32x2_t f = {lo, hi};
  if (FP16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2_t));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
}

// f over the lanes i, i ^ 16, i ^ 32 and i ^ 48, by swaps of rows between registers: a shuffle would stand in line behind every wave's reads of
// the tile.
template <class F>
__device__ __forceinline__ float over_rows(float v, F f) {
  const auto near = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(near[0]), __uint_as_float(near[1]));
  const auto far = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(far[0]), __uint_as_float(far[1]));
}

template <bool FP16>
__device__ __forceinline__ float elem_to_f32(uint16_t h) {
  return FP16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
}

// One workgroup per (batch, key/value head, split).  Wave w serves query head w % G and the
// columns [slice * D / CS, (slice + 1) * D / CS) of the output, slice = w / G: with few query
// heads per key/value head the output columns are split over CS waves (each repeats the cheap
// K Q^T) so that a SIMD has more than one wave to switch between.  Every launch has kThreads
// threads: waves beyond G * CS move tiles only.
template <int D, bool FP16, int CS, bool MASK, bool BLOCK>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_q16_kernel(KernelArgs<BLOCK> a) {
  constexpr int kCols = D / 16 / CS;          // 16-column chunks of the output per wave
  constexpr int P = D + kPadElems;            // row pitch of a tile in LDS, elements
  constexpr int kTileElems = kTileKeys * P;   // one K or V tile
  constexpr int kChunks = kTileKeys * D / 8;  // 16-byte pieces of a tile
  constexpr int kLoads = kChunks / kThreads;  // per thread: every launch has kThreads threads
  extern __shared__ __align__(16) uint16_t lds[];  // [2][K tile | V tile]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = a.ranges.quotient((int)blockIdx.x), split = (int)blockIdx.x - bh * a.splits;
  const int b = a.key_heads.quotient(bh), hk = bh - b * a.Hk;
  const int n_begin = split * a.keys_per_split;
  const int n_end = n_begin + a.keys_per_split < a.N ? n_begin + a.keys_per_split : a.N;
  // BLOCK: keys from here on are the block's own, which the cache does not hold yet; a last range of fewer than 16 keys
  // leaves some of them to the one before it.
  const int cached = BLOCK ? a.N - 16 : a.N;
  const bool has_block = BLOCK && n_end > cached;
  const int n_there = n_end < cached ? n_end : cached;  // (may be n_begin or less)
  const int full = !has_block ? n_end : n_begin < cached ? n_begin + (cached - n_begin) / kTileKeys * kTileKeys : n_begin;
  const int j = lane & 15, kb = lane >> 4;
  const bool computes = wave < a.G * CS;  // the other waves only move tiles
  int slice = 0, of_group = computes ? wave : 0;  // wave / G, wave % G
  while (of_group >= a.G) of_group -= a.G, ++slice;
  const int hq = hk * a.G + of_group;
  const size_t qrow = ((size_t)b * a.Hq + hq) * 16 + j;  // this lane's query

  const uint16_t* kbase = a.k + (size_t)b * a.k_batch_stride + (size_t)hk * a.k_head_stride;
  const uint16_t* vbase = a.v + (size_t)b * a.v_batch_stride + (size_t)hk * a.v_head_stride;

  // ---- tile movement: global -> registers -> LDS.  Two register stages: tile i + 1 goes from its
  // registers to LDS after the arithmetic of tile i, and the loads of tile i + 3 are issued to them at
  // once, ahead of the barrier.  Three tiles are on their way while the queries are prepared (two:
  // 32 716 keys of 8 x 256 60.4 us instead of 58.0, 14 016 of 8 x 128 23.0 instead of 21.7, 4 112 of 8 x 256 19.1
  // and 18.8; four and more in registers are slower again, 60.2, 25.1 and 21.2: a CU's first-level cache is
  // 32 KiB, as much as one tile of 256 columns; V read ahead of the softmax instead of behind it 62.5).  Nothing here is conditional: rows past
  // the end of the range repeat its last row (their scores are masked, their weights zero) and a
  // tile past the end is fetched and dropped, so that the number of loads in flight at every wait
  // is known when the kernel is compiled and a wait covers the older tile only. -----------------
  typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;  // a native vector: plain loads and stores
  struct Stage {
    u32x4_t k[kLoads], v[kLoads];
  };
  Stage stage0, stage1;
  auto fetch = [&](Stage& st, int n0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int c = tid + i * kThreads;
      const int key = c / (D / 8), piece = c % (D / 8);
      const int n = n0 + key < n_there ? n0 + key : n_there - 1;
      st.k[i] = *reinterpret_cast<const u32x4_t*>(kbase + (size_t)n * a.k_seq_stride + 8 * piece);
      st.v[i] = *reinterpret_cast<const u32x4_t*>(vbase + (size_t)n * a.v_seq_stride + 8 * piece);
    }
  };
  auto stash = [&](const Stage& st, int buf) __attribute__((always_inline)) {
    uint16_t* sk = lds + buf * 2 * kTileElems;
    uint16_t* sv = sk + kTileElems;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int c = tid + i * kThreads;
      const int key = c / (D / 8), piece = c % (D / 8);
      *reinterpret_cast<u32x4_t*>(sk + key * P + 8 * piece) = st.k[i];
      *reinterpret_cast<u32x4_t*>(sv + key * P + 8 * piece) = st.v[i];
    }
  };

  // ---- this wave's queries, as the B operand of K Q^T -----------------------------------------
  uint4 qreg[D / 32];
#pragma unroll
  for (int s = 0; s < D / 32; ++s) {
    const uint16_t* from = a.q + qrow * D;
    if constexpr (BLOCK) from = a.block.q + b * a.block.q_batch + j * a.block.q_row + (size_t)hq * (2 * D);
    qreg[s] = *reinterpret_cast<const uint4*>(from + 32 * s + 8 * kb);  // (waves that only move tiles: a head's, not looked at)
  }
  // (asked for ahead of the tiles: loads return in order, and the first product needs these)
  [[maybe_unused]] uint4 qw[BLOCK ? D / 32 : 1];
  if constexpr (BLOCK) {
#pragma unroll
    for (int s = 0; s < D / 32; ++s) qw[s] = *reinterpret_cast<const uint4*>(a.block.q_weight + 32 * s + 8 * kb);
  }

  fetch(stage0, n_begin);
  fetch(stage1, n_begin + kTileKeys);

  [[maybe_unused]] uint16_t* const block_k = lds + 4 * kTileElems;  // the block's own 16 rows
  [[maybe_unused]] uint16_t* const block_v = block_k + 16 * P;
  if constexpr (BLOCK) {
    // Norm and rotation of the queries by the waves that multiply with them, of the block's keys by the ranges that have some of
    // them, the last of which also writes them to the cache; all while the first tiles are on their way.  A launch of its own for it (attn_prepare_kernel,
    // whose bits these are) took 4 to 5 us and its place in the queue.  Here every range does it again, bound by its vector
    // instructions: 1.5 us of a launch with heads of 128, 3.2 of 256 (4.7 with one wave for all of a head's queries and the
    // powers computed by every thread).  Layer calls, us, before and with it: 4 112 keys of 8 x 256 48.5 -> 46.9, 32 716 92.3 ->
    // 89.1 (with the third tile on its way); of calls that the host bounds (five launches, now four) 9 152 keys of 8 x 128 43.3 -> 36.1, 2 343 of 2 x 256 43.1 -> 34.8.
    constexpr int PER = D / 64, kRowsPerWave = 16 / (kThreads / 64);
    const BlockArgs& p = a.block;
    const int half = p.half, pitch = half + kTurnPad;
    float2* const turn = reinterpret_cast<float2*>(lds + 5 * kTileElems);  // cosine and sine, [token][pair]
    float* const frequency = reinterpret_cast<float*>(turn + 16 * pitch);
    uint32_t k_raw[kRowsPerWave][PER], v_raw[kRowsPerWave][PER], kw_raw[PER];
    if (has_block) {
      load_adjacent_raw<PER>(p.k_weight, PER * lane, false, kw_raw);
#pragma unroll
      for (int u = 0; u < kRowsPerWave; ++u) {
        const int row = kRowsPerWave * wave + u;
        load_adjacent_raw<PER>(p.k + b * p.k_batch + row * p.k_row + (size_t)hk * D, PER * lane, false, k_raw[u]);
        load_adjacent_raw<PER>(p.v + b * p.v_batch + row * p.v_row + (size_t)hk * D, PER * lane, false, v_raw[u]);
      }
    }
    asm volatile("" ::: "memory");  // on their way before the angles
    if (tid < half) frequency[tid] = powf(p.base, -(float)tid * p.inv_half);
    __syncthreads();
    {
      const int shift = 31 - __builtin_clz(half), pair = tid & (half - 1);
      const float f = frequency[pair];
      for (int row = tid >> shift; row < 16; row += kThreads >> shift) {
        float2 t;
        sincosf((float)(a.N - 16 + row) * f, &t.y, &t.x);
        turn[row * pitch + pair] = t;
      }
    }
    // the first tile is there: room for the third, which comes while the queries are turned
    stash(stage0, 0);
    fetch(stage0, n_begin + 2 * kTileKeys);
    __syncthreads();
    if (computes) {
#pragma clang fp contract(off)
      constexpr int S = D / 32, H = 8 / PER;
      auto element = [](const uint4& v, int e) __attribute__((always_inline)) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        return elem_to_f32<FP16>((uint16_t)(e & 1 ? w[e >> 1] >> 16 : w[e >> 1]));
      };
      // the squares in the order in which a wave that has PER adjacent features a lane adds them up
      float part[S][H];
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int h = 0; h < H; ++h) {
          part[s][h] = 0.f;
#pragma unroll
          for (int e = 0; e < PER; ++e) {
            const float x = element(qreg[s], PER * h + e);
            part[s][h] += x * x;
          }
        }
#pragma unroll
      for (int step = S / 2; step >= 1; step /= 2)
#pragma unroll
        for (int s = 0; s < step; ++s)
#pragma unroll
          for (int h = 0; h < H; ++h) part[s][h] += part[s + step][h];
#pragma unroll
      for (int h = 0; h < H; ++h) part[0][h] += __shfl_xor(part[0][h], 32, 64);
#pragma unroll
      for (int h = 0; h < H; ++h) part[0][h] += __shfl_xor(part[0][h], 16, 64);
#pragma unroll
      for (int step = H / 2; step >= 1; step /= 2)
#pragma unroll
        for (int h = 0; h < step; ++h) part[0][h] += part[0][h + step];
      const float inv_rms = 1.0f / sqrtf(part[0][0] * (1.0f / (float)D) + p.q_eps);
      // The waves that share a head each take kWords of the four words of every piece, and meet in the second tile's place.
      constexpr int kWords = 4 / CS;
      uint32_t mine[S][kWords];
      auto word = [](const uint4& v, int w) __attribute__((always_inline)) { return w == 0 ? v.x : w == 1 ? v.y : w == 2 ? v.z : v.w; };
      auto low = [](uint32_t w) __attribute__((always_inline)) { return elem_to_f32<FP16>((uint16_t)w); };
      auto high = [](uint32_t w) __attribute__((always_inline)) { return elem_to_f32<FP16>((uint16_t)(w >> 16)); };
      auto rounded = [](float x, float y) __attribute__((always_inline)) {
        return FP16 ? pack2<FP16>(in_full(x), in_full(y)) : pack2<FP16>(x, y);
      };
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int i = 0; i < kWords; ++i) {
          uint32_t x = word(qreg[s], i), w = word(qw[s], i);
#pragma unroll
          for (int c = 1; c < CS; ++c) {
            uint32_t other_x = word(qreg[s], kWords * c + i), other_w = word(qw[s], kWords * c + i);
            asm("" : "+v"(other_x), "+v"(other_w));  // (a choice of values: of addresses, the pieces would go to memory)
            x = slice == c ? other_x : x, w = slice == c ? other_w : w;
          }
          mine[s][i] = rounded(low(x) * inv_rms * low(w), high(x) * inv_rms * high(w));
        }
      // features i and i + half, in pieces s and s + half / 32 of one lane
      auto rotate = [&](auto apart) __attribute__((always_inline)) {
        constexpr int A = decltype(apart)::value;
        if constexpr (2 * A <= S) {
#pragma unroll
          for (int s = 0; s < A; ++s)
#pragma unroll
            for (int i = 0; i < kWords; ++i) {
              // cosine and sine of two pairs
              const f32x4_t t = *reinterpret_cast<const f32x4_t*>(turn + j * pitch + 32 * s + 8 * kb + 2 * (kWords * slice + i));
              const uint32_t xw = mine[s][i], yw = mine[s + A][i];
              const float x0 = low(xw), x1 = high(xw), y0 = low(yw), y1 = high(yw);
              mine[s][i] = rounded(x0 * t[0] - y0 * t[1], x1 * t[2] - y1 * t[3]);
              mine[s + A][i] = rounded(x0 * t[1] + y0 * t[0], x1 * t[3] + y1 * t[2]);
            }
        }
      };
      if (half == 32) rotate(std::integral_constant<int, 1>{});
      else if (half == 64) rotate(std::integral_constant<int, 2>{});
      else rotate(std::integral_constant<int, 4>{});
      uint32_t* const shared = reinterpret_cast<uint32_t*>(lds + 2 * kTileElems) + (of_group * S * 64 + lane) * 4;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if constexpr (CS == 1) qreg[s] = uint4{mine[s][0], mine[s][1 % kWords], mine[s][2 % kWords], mine[s][3 % kWords]};
        else if constexpr (CS == 2) *reinterpret_cast<uint2*>(shared + 256 * s + 2 * slice) = uint2{mine[s][0], mine[s][1 % kWords]};
        else shared[256 * s + slice] = mine[s][0];
      }
    }
    if constexpr (CS > 1) {
      __syncthreads();
      if (computes) {
#pragma unroll
        for (int s = 0; s < D / 32; ++s) qreg[s] = reinterpret_cast<const uint4*>(lds + 2 * kTileElems)[(of_group * (D / 32) + s) * 64 + lane];
      }
    }
    if (has_block) {
      constexpr int dt = FP16 ? DFLASH_FP16 : DFLASH_BF16;
      const int c = PER * lane;
      const bool rotates = c < 2 * half, upper = c >= half;
      const int other = rotates ? (upper ? lane - half / PER : lane + half / PER) : lane;
      float w[PER];
      unpack_adjacent<PER>(kw_raw, dt, w);
#pragma unroll
      for (int u = 0; u < kRowsPerWave; ++u) {
        const int row = kRowsPerWave * wave + u;
        float x[PER], cs[PER], sn[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
          const float2 t = turn[row * pitch + (rotates ? (upper ? c - half : c) + e : 0)];
          cs[e] = t.x, sn[e] = t.y;
        }
        unpack_adjacent<PER>(k_raw[u], dt, x);
        norm_and_turn<PER>(x, w, p.k_eps, cs, sn, rotates, upper, other, dt);
        const long long at = b * a.k_batch_stride + hk * a.k_head_stride + (a.N - 16 + row) * a.k_seq_stride + c;
        const long long vat = b * a.v_batch_stride + hk * a.v_head_stride + (a.N - 16 + row) * a.v_seq_stride + c;
        store_adjacent<PER>(block_k, (size_t)(row * P + c), dt, x);
        store_raw<PER>(block_v + row * P + c, v_raw[u]);
        if (split == a.splits - 1) {
          store_adjacent<PER>(p.k_cache, (size_t)at, dt, x);
          store_raw<PER>(p.v_cache + vat, v_raw[u]);
        }
      }
    }
  }

  f32x4_t O[kCols];
#pragma unroll
  for (int c = 0; c < kCols; ++c) O[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = kMasked, l_run = 0.f;  // l_run: this lane's keys only, merged at the end

  // OWN: a tile with keys of the block, which are read where they were prepared.  Where they take their places among the cached ones,
  // ranges and tiles are those of a block whose rows were in the cache before the launch, and so are the results' bits.
  auto compute_tile = [&](const uint16_t* sk, int n0, auto own) __attribute__((always_inline)) {
    constexpr bool OWN = decltype(own)::value;
    if (computes) {
      const uint16_t* sv = sk + kTileElems;
      auto row_of = [&](const uint16_t* tile, const uint16_t* block, int i) __attribute__((always_inline)) {  // of key n0 + i
        if constexpr (!OWN) return tile + i * P;
        const int at = n0 + i - cached;
        return at < 0 ? tile + i * P : block + (at < 16 ? at : 15) * P;  // (behind the last key: that one, not counted)
      };
      // S^T = K Q^T for the two 16-key halves of the tile
      // (all reads of the tile are issued before the first product: one LDS latency, not sixteen)
      uint4 kf[2][D / 32];
#pragma unroll
      for (int s = 0; s < D / 32; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) kf[t][s] = *reinterpret_cast<const uint4*>(row_of(sk, block_k, 16 * t + j) + 32 * s + 8 * kb);
      f32x4_t st[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int s = 0; s < D / 32; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) st[t] = mfma32<FP16>(kf[t][s], qreg[s], st[t]);
      // scores of query j for keys n0 + 16 t + 4 kb + r
      float x[8];
      bool use[8];
      float m_tile = kMasked;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = n0 + 16 * t + 4 * kb + r;
          bool ok = n < n_end && n <= a.N - 16 + j;
          float s = st[t][r] * a.scale;
          if (MASK && ok) {
            const float mv = elem_to_f32<FP16>(a.mask[qrow * a.N + n]);
            ok = mv >= a.lowest;
            s += mv;
          }
          use[4 * t + r] = ok;
          x[4 * t + r] = ok ? s : kMasked;
          m_tile = fmaxf(m_tile, x[4 * t + r]);
        }
      }
      m_tile = over_rows(m_tile, [](float x, float y) { return fmaxf(x, y); });
      const float m_new = fmaxf(m_run, m_tile);
      const float factor = __expf(m_run - m_new);  // 1 while nothing has been seen (both masked)
      float p[8], sum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = use[e] ? __expf(x[e] - m_new) : 0.f;
        sum += p[e];
      }
      l_run = l_run * factor + sum;
      m_run = m_new;
      if (__any(factor != 1.f)) {
#pragma unroll
        for (int c = 0; c < kCols; ++c) O[c] *= factor;
      }
      const uint4 pb = {pack2<FP16>(p[0], p[1]), pack2<FP16>(p[2], p[3]), pack2<FP16>(p[4], p[5]),
                        pack2<FP16>(p[6], p[7])};
      // O^T += V^T P^T, 16 columns of V at a time
      const int src = lane & 15;  // source lane inside the group of 16: key 4 kb + src / 4, columns 4 (src % 4) ..+3
      const int piece = 4 * (src & 3) + 16 * kCols * slice;
      const uint16_t* const vlow = row_of(sv, block_v, 4 * kb + (src >> 2)) + piece;
      const uint16_t* const vhigh = row_of(sv, block_v, 16 + 4 * kb + (src >> 2)) + piece;
      typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
      s16x4_t lo[kCols], hi[kCols];
#pragma unroll
      for (int c = 0; c < kCols; ++c) {
        lo[c] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vlow + 16 * c));
        hi[c] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vhigh + 16 * c));
      }
#pragma unroll
      for (int c = 0; c < kCols; ++c) {
        const uint2 lo2 = __builtin_bit_cast(uint2, lo[c]), hi2 = __builtin_bit_cast(uint2, hi[c]);
        O[c] = mfma32<FP16>(uint4{lo2.x, lo2.y, hi2.x, hi2.y}, pb, O[c]);
      }
    }

  };

  if constexpr (!BLOCK) {
    stash(stage0, 0);
    fetch(stage0, n_begin + 2 * kTileKeys);
  }
  __syncthreads();
  for (int n0 = n_begin; n0 < full; n0 += 2 * kTileKeys) {
    // even tile in buffer 0, the next one in stage 1, the one after it on its way to stage 0
    compute_tile(lds, n0, std::false_type{});
    stash(stage1, 1);
    fetch(stage1, n0 + 3 * kTileKeys);
    __syncthreads();
    if (n0 + kTileKeys >= full) break;
    compute_tile(lds + 2 * kTileElems, n0 + kTileKeys, std::false_type{});
    stash(stage0, 0);
    fetch(stage0, n0 + 4 * kTileKeys);
    __syncthreads();
  }
  if constexpr (BLOCK) {
    if (has_block) {
      // the first of these tiles may begin with cached keys and is in the buffer of its turn; a second one is the block's alone
      const uint16_t* const from = lds + ((full - n_begin) / kTileKeys & 1) * 2 * kTileElems;
#pragma unroll 1
      for (int n0 = full; n0 < n_end; n0 += kTileKeys) compute_tile(from, n0, std::true_type{});
    }
  }

  if (!computes) return;
  l_run = over_rows(l_run, [](float x, float y) { return x + y; });
  // accumulator r of chunk c is column 16 (kCols slice + c) + 4 kb + r of query j
  const int col0 = 16 * kCols * slice + 4 * kb;
  if (a.splits == 1) {
    const float inv = l_run > 0.f ? 1.f / l_run : 1.f;
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const uint2 o = {pack2<FP16>(O[c][0] * inv, O[c][1] * inv), pack2<FP16>(O[c][2] * inv, O[c][3] * inv)};
      *reinterpret_cast<uint2*>(a.out + qrow * D + col0 + 16 * c) = o;
    }
  } else {
    const size_t prow = (size_t)split * a.B * a.Hq * 16 + qrow;
#pragma unroll
    for (int c = 0; c < kCols; ++c)
      *reinterpret_cast<uint2*>(a.part_o + prow * D + col0 + 16 * c) =
          uint2{pack2<FP16>(O[c][0], O[c][1]), pack2<FP16>(O[c][2], O[c][3])};
    if (kb == 0 && slice == 0) *reinterpret_cast<f32x2_t*>(a.part_ml + prow * 2) = f32x2_t{m_run, l_run};
  }
}

// Second pass: one workgroup of 256 threads per query row.  Thread (g, c) adds the partial
// outputs of the splits s = g, g + 4, ... for 4 output columns; the weights exp(m_s - m) and the
// total sum are worked out once, by the first wave.
constexpr int kMaxSplits = 256;
template <bool FP16>
__global__ __launch_bounds__(256) void sdpa_q16_merge_kernel(SdpaArgs a, int D) {
  __shared__ float weight[kMaxSplits];
  __shared__ float total;
  __shared__ f32x4_t acc[4][64];
  const size_t row = blockIdx.x;  // (b * Hq + hq) * 16 + i
  const size_t rows = (size_t)a.B * a.Hq * 16;
  const int tid = threadIdx.x, c4 = tid & 63, g = tid >> 6;
  const bool col = 4 * c4 < D;
  // Group g adds up splits g, g + 4, ...; eight of them per round.  The first round's partial
  // outputs are asked for before anything else, and every round asks for all eight before it
  // uses one: a split's answer takes a microsecond, and there are up to 64 per group.
  constexpr int kRound = 8;
  uint2 h[kRound];
  auto issue_round = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kRound; ++j) {
      const int s = s0 + 4 * j;
      h[j] = uint2{0u, 0u};
      if (col && s < a.splits) h[j] = *reinterpret_cast<const uint2*>(a.part_o + ((size_t)s * rows + row) * D + 4 * c4);
    }
  };
  issue_round(g);
  // (b, hq, i) of the row; the gate is asked for with the partial results
  const int i = (int)blockIdx.x % 16, head = (int)blockIdx.x / 16, b = a.heads.quotient(head), hq = head - b * a.Hq;
  uint2 gate = uint2{0u, 0u};
  if (a.gate != nullptr && g == 0 && col)
    gate = *reinterpret_cast<const uint2*>(a.gate + b * a.gate_batch_stride + i * a.gate_row_stride + (size_t)hq * 2 * D + D + 4 * c4);
  if (tid < 64) {
    f32x2_t ml[kMaxSplits / 64];
#pragma unroll
    for (int j = 0; j < kMaxSplits / 64; ++j) {
      const int s = tid + 64 * j;
      ml[j] = f32x2_t{kMasked, 0.f};
      if (s < a.splits) ml[j] = *reinterpret_cast<const f32x2_t*>(a.part_ml + ((size_t)s * rows + row) * 2);
    }
    float m = kMasked;
#pragma unroll
    for (int j = 0; j < kMaxSplits / 64; ++j) m = fmaxf(m, ml[j][0]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    float l = 0.f;
#pragma unroll
    for (int j = 0; j < kMaxSplits / 64; ++j) {
      const int s = tid + 64 * j;
      if (s < a.splits) {
        const float w = __expf(ml[j][0] - m);
        weight[s] = w;
        l += w * ml[j][1];
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) l += __shfl_xor(l, off, 64);
    if (tid == 0) total = l;
  }
  __syncthreads();
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = g; s0 < a.splits; s0 += 4 * kRound) {
    if (s0 != g) issue_round(s0);
#pragma unroll
    for (int j = 0; j < kRound; ++j) {
      const int s = s0 + 4 * j;
      if (s < a.splits) {
        const f32x4_t v = {elem_to_f32<FP16>((uint16_t)h[j].x), elem_to_f32<FP16>((uint16_t)(h[j].x >> 16)),
                           elem_to_f32<FP16>((uint16_t)h[j].y), elem_to_f32<FP16>((uint16_t)(h[j].y >> 16))};
        o += v * weight[s];
      }
    }
  }
  acc[g][c4] = o;
  __syncthreads();
  if (g == 0 && col) {
    o = acc[0][c4] + acc[1][c4] + acc[2][c4] + acc[3][c4];
    const float inv = total > 0.f ? 1.f / total : 1.f;
    uint2 packed = {pack2<FP16>(o[0] * inv, o[1] * inv), pack2<FP16>(o[2] * inv, o[3] * inv)};
    size_t to = row;
    if (a.gate != nullptr) {
      // output * sigmoid(gate) as the array operators give it: output, sigmoid and product each of the array's type
      const uint32_t gw[4] = {gate.x & 0xFFFFu, gate.x >> 16, gate.y & 0xFFFFu, gate.y >> 16};
      const uint32_t ow[4] = {packed.x & 0xFFFFu, packed.x >> 16, packed.y & 0xFFFFu, packed.y >> 16};
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sig = sigmoid_of_half(elem_to_f32<FP16>((uint16_t)gw[e]));  // the bits of attn_gate_kernel
        y[e] = elem_to_f32<FP16>((uint16_t)ow[e]) * elem_to_f32<FP16>((uint16_t)pack2<FP16>(sig, 0.f));
      }
      packed = uint2{pack2<FP16>(y[0], y[1]), pack2<FP16>(y[2], y[3])};
      to = ((size_t)b * 16 + i) * a.Hq + hq;
    }
    *reinterpret_cast<uint2*>(a.out + to * D + 4 * c4) = packed;
  }
}

int pick_splits(int B, int Hk, int N, int* keys_per_split) {
  // About one workgroup per compute unit, and never less than 128 keys per split: every split
  // adds B * Hq * 16 * (2 D + 8) bytes of partial results, written once and read once.
  // DFLASH_OPT_SDPA_SPLITS = n asks for n ranges instead (tests)
  const int forced = option(DFLASH_OPT_SDPA_SPLITS);
  int want = forced > 0 ? forced : (256 + B * Hk - 1) / (B * Hk);
  const int most = (N + 127) / 128;
  if (want > most) want = most;
  if (want > kMaxSplits) want = kMaxSplits;
  if (want < 1) want = 1;
  int per = (N + want - 1) / want;
  per = (per + kTileKeys - 1) / kTileKeys * kTileKeys;
  *keys_per_split = per;
  return (N + per - 1) / per;  // no empty split
}

size_t partial_bytes(int splits, int B, int Hq, int D) {
  return splits == 1 ? 0 : (size_t)splits * B * Hq * 16 * (D * sizeof(uint16_t) + 2 * sizeof(float));
}

}  // namespace
}  // namespace dflash

extern "C" size_t dflash_sdpa_q16_workspace_bytes(int B, int Hq, int Hk, int N, int D) {
  using namespace dflash;
  if (B <= 0 || Hq <= 0 || Hk <= 0 || N <= 0 || D <= 0) return 0;
  int per = 0;
  return partial_bytes(pick_splits(B, Hk, N, &per), B, Hq, D);
}

extern "C" size_t dflash_attn_block_workspace_bytes(int B, int Hq, int Hk, int N, int D) {
  using namespace dflash;
  return N > 16 ? dflash_sdpa_q16_workspace_bytes(B, Hq, Hk, N, D) : 0;
}

namespace dflash {
namespace {
int sdpa_launch(const void* q, const void* k, const void* v, const void* mask, const void* gate, void* out,
                void* workspace, size_t workspace_bytes, int B, int Hq, int Hk, int N, int D,
                long long k_batch_stride, long long k_head_stride, long long k_seq_stride,
                long long v_batch_stride, long long v_head_stride, long long v_seq_stride,
                long long gate_batch_stride, long long gate_row_stride, float scale, int dtype, void* stream,
                const BlockArgs* block = nullptr) {
  DFLASH_REQUIRE(q && k && v && out, DFLASH_ERR_ARG, "dflash_sdpa_q16: null operand");
  DFLASH_REQUIRE(dtype == DFLASH_BF16 || dtype == DFLASH_FP16, DFLASH_ERR_ARG,
                 "dflash_sdpa_q16: bf16 or fp16 only");
  DFLASH_REQUIRE(D == 128 || D == 256, DFLASH_ERR_SHAPE, "dflash_sdpa_q16: head dim %d (128 or 256)", D);
  DFLASH_REQUIRE(B > 0 && Hq > 0 && Hk > 0 && N >= 16 && Hq % Hk == 0 && Hq / Hk <= 8, DFLASH_ERR_SHAPE,
                 "dflash_sdpa_q16: B %d, Hq %d, Hk %d, N %d (Hq a multiple of Hk, at most 8 times; N >= 16)", B, Hq,
                 Hk, N);
  DFLASH_REQUIRE(k_seq_stride >= D && v_seq_stride >= D && k_seq_stride % 8 == 0 && v_seq_stride % 8 == 0 &&
                     k_head_stride % 8 == 0 && v_head_stride % 8 == 0 && k_batch_stride % 8 == 0 &&
                     v_batch_stride % 8 == 0,
                 DFLASH_ERR_SHAPE, "dflash_sdpa_q16: strides must keep rows 16-byte aligned");
  DFLASH_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) % 16) == 0, DFLASH_ERR_ARG,
                 "dflash_sdpa_q16: operands must be 16-byte aligned");
  DFLASH_REQUIRE((long long)B * Hq * 16 < (1ll << 31) && (long long)B * Hk * ((N + 127) / 128) < (1ll << 31),
                 DFLASH_ERR_SHAPE, "dflash_sdpa_q16: too many rows");

  KernelArgs<true> a;
  a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v; a.mask = (const uint16_t*)mask;
  a.out = (uint16_t*)out;
  a.k_batch_stride = k_batch_stride; a.k_head_stride = k_head_stride; a.k_seq_stride = k_seq_stride;
  a.v_batch_stride = v_batch_stride; a.v_head_stride = v_head_stride; a.v_seq_stride = v_seq_stride;
  a.B = B; a.Hq = Hq; a.Hk = Hk; a.N = N; a.G = Hq / Hk;
  a.splits = pick_splits(B, Hk, N, &a.keys_per_split);
  if (block) a.block = *block;
  a.ranges = Divisor::of(a.splits); a.key_heads = Divisor::of(Hk); a.heads = Divisor::of(Hq);
  a.scale = scale;
  a.lowest = dtype == DFLASH_FP16 ? -65504.0f : -3.3895313892515355e38f;
  a.gate = (const uint16_t*)gate;
  a.gate_batch_stride = gate_batch_stride; a.gate_row_stride = gate_row_stride;
  DFLASH_REQUIRE(!gate || a.splits > 1, DFLASH_ERR_SHAPE, "dflash_sdpa_q16_gated: the gate rides on the merge of key ranges");
  a.part_o = nullptr;
  a.part_ml = nullptr;
  if (a.splits > 1) {
    const size_t need = partial_bytes(a.splits, B, Hq, D);
    DFLASH_REQUIRE(workspace && workspace_bytes >= need && ((uintptr_t)workspace % 16) == 0, DFLASH_ERR_WORKSPACE,
                   "dflash_sdpa_q16: workspace of %zu bytes needed, %zu given", need,
                   workspace ? workspace_bytes : (size_t)0);
    a.part_ml = (float*)workspace;   // [splits, rows, 2] fp32 first: keeps both arrays 16-byte aligned
    a.part_o = (uint16_t*)(a.part_ml + (size_t)a.splits * B * Hq * 16 * 2);
  }

  hipStream_t s = (hipStream_t)stream;
  // column split: as many waves as fit eight, in powers of two
  const int cs = a.G <= 2 ? 4 : a.G <= 4 ? 2 : 1;
  const int tiles = block ? 5 : 4;  // (a block's rows: half a tile of keys, half of values)
  const size_t lds_bytes = (size_t)tiles * kTileKeys * (D + kPadElems) * sizeof(uint16_t) +
                           (block ? turn_bytes(block->half) : 0);
  const size_t lds_most = (size_t)tiles * kTileKeys * (D + kPadElems) * sizeof(uint16_t) +
                          (block ? turn_bytes(D / 2) : 0);
  const bool f16 = dtype == DFLASH_FP16;
#define DFLASH_SDPA_ROW(D_, F_, M_, B_)                                                                        \
  {(const void*)sdpa_q16_kernel<D_, F_, 1, M_, B_>, (const void*)sdpa_q16_kernel<D_, F_, 2, M_, B_>, \
   (const void*)sdpa_q16_kernel<D_, F_, 4, M_, B_>}
#define DFLASH_SDPA_FORMS(D_, F_) {DFLASH_SDPA_ROW(D_, F_, false, false), DFLASH_SDPA_ROW(D_, F_, true, false), DFLASH_SDPA_ROW(D_, F_, false, true)}
  static const void* const table[2][2][3][3] = {{DFLASH_SDPA_FORMS(128, false), DFLASH_SDPA_FORMS(128, true)},
                                                {DFLASH_SDPA_FORMS(256, false), DFLASH_SDPA_FORMS(256, true)}};
#undef DFLASH_SDPA_FORMS
#undef DFLASH_SDPA_ROW
  const int form = block ? 2 : mask != nullptr ? 1 : 0;
  const int ics = cs == 1 ? 0 : cs == 2 ? 1 : 2;
  void* args[] = {&a};
  const int slot = current_device_slot();
  {
    const void* fn = table[D == 256][f16][form][ics];
    // the attribute belongs to the device's copy of the kernel: once per device and kernel
    static bool attr_set[kMaxDevices][2][2][3][3] = {};
    bool& set = attr_set[slot][D == 256][f16][form][ics];
    if (!set || slot == kMaxDevices - 1) {
      DFLASH_HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_most));
      set = true;
    }
    DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)(B * Hk * a.splits)), dim3(kThreads), args, lds_bytes, s));
  }
  if (a.splits > 1) {
    if (dtype == DFLASH_FP16) {
      hipLaunchKernelGGL(sdpa_q16_merge_kernel<true>, dim3((unsigned)(B * Hq * 16)), dim3(256), 0, s, (const SdpaArgs&)a, D);
    } else {
      hipLaunchKernelGGL(sdpa_q16_merge_kernel<false>, dim3((unsigned)(B * Hq * 16)), dim3(256), 0, s, (const SdpaArgs&)a, D);
    }
    DFLASH_HIP_OK(hipGetLastError());
  }
  return DFLASH_OK;
}
}  // namespace
}  // namespace dflash

extern "C" int dflash_sdpa_q16(const void* q, const void* k, const void* v, const void* mask, void* out,
                               void* workspace, size_t workspace_bytes, int B, int Hq, int Hk, int N, int D,
                               long long k_batch_stride, long long k_head_stride, long long k_seq_stride,
                               long long v_batch_stride, long long v_head_stride, long long v_seq_stride,
                               float scale, int dtype, void* stream) {
  return dflash::sdpa_launch(q, k, v, mask, nullptr, out, workspace, workspace_bytes, B, Hq, Hk, N, D, k_batch_stride,
                             k_head_stride, k_seq_stride, v_batch_stride, v_head_stride, v_seq_stride, 0, 0, scale, dtype, stream);
}

// A launch of its own for the gate (dflash_attn_gate) cost 4 us on the device and 10 us of host time behind an attention
// of 15 us (4 112 keys): layer call 92 -> 86 us, over 32 716 keys 99 -> 96 us.
extern "C" int dflash_sdpa_q16_gated(const void* q, const void* k, const void* v, const void* mask, const void* gate,
                                     void* out, void* workspace, size_t workspace_bytes, int B, int Hq, int Hk, int N,
                                     int D, long long k_batch_stride, long long k_head_stride, long long k_seq_stride,
                                     long long v_batch_stride, long long v_head_stride, long long v_seq_stride,
                                     long long gate_batch_stride, long long gate_row_stride, float scale, int dtype,
                                     void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(gate, DFLASH_ERR_ARG, "dflash_sdpa_q16_gated: null gate");
  DFLASH_REQUIRE(gate_batch_stride >= 0 && gate_row_stride >= 0 &&
                     (((uintptr_t)gate | (uintptr_t)(gate_batch_stride * 2) | (uintptr_t)(gate_row_stride * 2)) % 8) == 0,
                 DFLASH_ERR_ARG, "dflash_sdpa_q16_gated: rows of the gate must be 8-byte aligned");
  return sdpa_launch(q, k, v, mask, gate, out, workspace, workspace_bytes, B, Hq, Hk, N, D, k_batch_stride, k_head_stride,
                     k_seq_stride, v_batch_stride, v_head_stride, v_seq_stride, gate_batch_stride, gate_row_stride, scale, dtype,
                     stream);
}

extern "C" int dflash_attn_block(const dflash_attn_block_args* args, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(args, DFLASH_ERR_ARG, "dflash_attn_block: null arguments");
  const dflash_attn_block_args& p = *args;
  DFLASH_REQUIRE(p.q && p.k && p.v && p.q_weight && p.k_weight && p.k_cache && p.v_cache && p.out, DFLASH_ERR_ARG, "dflash_attn_block: null operand");
  DFLASH_REQUIRE(p.N > 16, DFLASH_ERR_SHAPE, "dflash_attn_block: no keys before the block (N %d)", p.N);
  DFLASH_REQUIRE(p.rope_dims == 64 || p.rope_dims == 128 || (p.rope_dims == 256 && p.D == 256), DFLASH_ERR_SHAPE,
                 "dflash_attn_block: %d rotated features of %d (64, 128 or 256)", p.rope_dims, p.D);
  const long long rows[] = {p.q_batch, p.q_row, p.k_batch, p.k_row, p.v_batch, p.v_row};
  uintptr_t bits = (uintptr_t)p.q | (uintptr_t)p.k | (uintptr_t)p.v | (uintptr_t)p.q_weight | (uintptr_t)p.k_weight;
  for (long long r : rows) {
    DFLASH_REQUIRE(r >= 0, DFLASH_ERR_SHAPE, "dflash_attn_block: negative stride");
    bits |= (uintptr_t)r * 2;
  }
  DFLASH_REQUIRE(bits % 16 == 0, DFLASH_ERR_ARG, "dflash_attn_block: operands and rows must be 16-byte aligned");
  BlockArgs b;
  b.q = (const uint16_t*)p.q; b.k = (const uint16_t*)p.k; b.v = (const uint16_t*)p.v;
  b.q_batch = p.q_batch; b.q_row = p.q_row; b.k_batch = p.k_batch; b.k_row = p.k_row; b.v_batch = p.v_batch; b.v_row = p.v_row;
  b.q_weight = (const uint16_t*)p.q_weight; b.k_weight = (const uint16_t*)p.k_weight;
  b.k_cache = (uint16_t*)p.k_cache; b.v_cache = (uint16_t*)p.v_cache;
  b.half = p.rope_dims / 2;
  b.q_eps = p.q_eps; b.k_eps = p.k_eps; b.base = p.rope_base; b.inv_half = 1.0f / (float)b.half;
  return sdpa_launch(p.q, p.k_cache, p.v_cache, nullptr, p.q, p.out, p.workspace, p.workspace_bytes, p.B, p.Hq, p.Hk, p.N, p.D,
                     p.k_cache_batch, p.k_cache_head, p.k_cache_row, p.v_cache_batch, p.v_cache_head, p.v_cache_row, p.q_batch,
                     p.q_row, p.scale, p.dtype, stream, &b);
}
