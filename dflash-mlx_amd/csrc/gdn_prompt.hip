// GatedDeltaNet forward over a prompt (T > 16 tokens, bf16 q / k / v, one gate per head) for gfx950.
//
// The recurrence of gdn_forward.hip (dflash_mlx/kernels.py:12-127) is sequential in t, and a kernel that
// walks it token by token takes microseconds per token.  Here the tokens go through in chunks of 32 in closed
// form.  With c_t = prod_{u<=t} g_u inside the chunk, L[t][s] = beta_t (c_t/c_s)(k_s.k_t) for s < t and
// Lq[t][s] = (c_t/c_s)(k_s.q_t) for s <= t (masked and missing tokens: g = 1, beta = 0),
//     Delta = M' (V - c U),   M' = (I + L)^-1 diag(beta),   U = K S0^T
//     Y     = c (Q S0^T) + Lq Delta
//     S^T   = c_T S0^T + K^T diag(c_T/c_s) Delta,
// a chunk needs the state only in two products with it and one update of it.
//
//  * gdn_chunk_kernel, four waves per (slot, chunk, head), computes what does not depend on the state: M' and
//    Lq, in the register order the other kernel multiplies them in, and K^T likewise.  All chunks at once.
//  * gdn_prompt_kernel, one workgroup per (slot, head, 16 rows of the state), walks the chunks.  Rows of S are
//    independent, so 32 heads of 128 x 128 fill 256 compute units with one workgroup each, and what bounds
//    the kernel is its chain of dependent steps.  Nothing in it crosses lanes: the accumulators of U^T, Delta^T and S^T (a
//    lane holds four consecutive rows of one column) are read as the B operand of the next product with k in the order the
//    lane happens to have it, and the A operands (M', Lq, K^T) were laid out in that order.
//  * Where that leaves the chip with one wave per compute unit, a row's elements are divided among as many waves as it has
//    32ths: each cuts its part of S into pieces, multiplies and updates it, and the parts of U and Q S0^T meet in LDS,
//    one barrier per chunk.  Delta is computed by all of them, from the same sums in the same order, Y by one each.
//  * fp32 factors (S, V - c U, Delta, M', Lq) are cut into three bf16 pieces (24 bits, exact); products with bf16
//    K and Q take three matrix-core passes, products of two fp32 factors the six of relative size 2^-16 and up.
//    The result carries fp32 accuracy, as the step-by-step kernel's does.
//  * The operands of the next chunk are loaded into the registers of the present one as soon as these have
//    been used for the last time; 1 or 2 waves per SIMD have registers for all of them.
//  * The closed form is for finite numbers: in a product over all tokens of a chunk, a NaN or an infinity meets the
//    zeros of M' and Lq and spoils tokens and rows of the state that it must not reach, and products of k with k
//    may overflow where the recurrence does not.  Both kernels look at what they computed (a sum of 0 x stays zero
//    as long as every x is finite), and such a chunk is walked token by token instead, by the same wave.  What a masked
//    token holds never enters a product: its rows of K and Q are zeros, its element of V - c U as well.
// A 16-bit state is carried in fp32 and rounded once, at the end.
//
// Measured, 1024 tokens, 16 / 32 heads of 128 x 128: 12.5 + 51 us (64 with one wave per 16 rows), against 123.7 ms with one
// workgroup per head that kept S in memory (the step-by-step kernel held 41 tokens at most); 678 tokens of 16 heads both kernels
// 46 us (55).  What the second kernel is bound by is its chain.  One wave: 4560 cycles (2 us) per chunk by its counters, 605
// vector instructions (53 %), 96 matrix instructions (34 %; 72 of them with S), waits 16 %.  Four: 3500 cycles, 315 vector and
// 36 matrix instructions a wave; with no loads in the loop at all it takes 2900, the rest is the hand-over and results that the next
// instruction waits for.  Chunks of
// 32 and not 16: cutting S into pieces (176 vector instructions) is paid per chunk, and a matrix instruction
// of depth 32 in the update is filled; 64 would need more registers than a wave has.  The look for numbers that are not
// finite costs 0.3 % of a layer call, a chunk token by token what 32 steps of one wave cost.
#include "gdn_device.h"

#include <type_traits>

namespace dflash {
namespace prompt {

constexpr int kChunk = 32;
constexpr int kMatBytes = 2 * 3 * 1024;                // [tile of 16 rows][piece][lane] 16 bytes
constexpr int kHeadBytes = 2 * kMatBytes + 3 * kChunk * 4;  // M', Lq, then per token c (0 if masked) and c_T / c_s, then kTail:
constexpr int kTail = 2 * kChunk;                      // four words: c_T, 0 or (numbers that are not finite) NaN, one bit per token that counts, -
constexpr int kPitch = 36;                             // floats per row of the 32 x 32 matrices in LDS
// Up to as many (head, 16 rows) as there are compute units, the 32ths of a row on a wave each.  With more of them the units
// are shared, and what the waves of a row do twice (Delta, the pieces of it) costs more than their chain is shorter: us per
// 1024 tokens with the chunk kernel, one wave and four, 32 heads of 128 x 128 78 and 66, 48 heads 88 and 90, 64 heads 89 and 94.
constexpr int kSpread = 256;

struct Args {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const void* g;
  const void* beta;
  const void* state_in;  // null: zeros
  void* state_out;
  uint16_t* y;
  float* tape;  // may be null
  const uint8_t* mask;
  char* work;
  int slots, T, chunks, Hk, Hv, Dv;
  int g_dtype, beta_dtype, state_dtype;
};

// Token (row 0 .. 31 of a chunk) that element j = 0 .. 7 of lane group kq holds in an operand of depth 32:
// accumulators of the two 16-row tiles, one after the other.
__device__ __forceinline__ int token_of(int kq, int j) { return 16 * (j >> 2) + 4 * kq + (j & 3); }
// dk that row i of 16-row tile c of S^T stands for: tiles 2C and 2C + 1 of a lane are 8 consecutive dk.
__device__ __forceinline__ int dk_of(int c, int i) { return 32 * (c >> 1) + 8 * (i >> 2) + 4 * (c & 1) + (i & 3); }

__device__ __forceinline__ f32x4_t mfma(uint4 a, const uint32_t (&b)[4], f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, uint4{b[0], b[1], b[2], b[3]}), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Raw buffer descriptor: 32-bit byte offsets, accesses from `bytes` on read zero and write nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
}

template <int DK>
__device__ __forceinline__ size_t chunk_bytes(const Args& a) {
  return (size_t)a.Hv * kHeadBytes + (size_t)a.Hk * (kChunk * DK * 2);
}

// Four waves on a chunk of a head.  What bounds a call of few chunks is the chain of one: a wave by itself took 12 us, its products, the 32
// steps of the ratios, 32 of the inverse and K^T out of LDS one after the other.  Here the products of K with K and Q are divided,
// two waves make the entries of 16 tokens each while the other two turn K, and the inverse is one of two 16 x 16 triangles side by
// side with the block below them from two products: X21 = -X22 (L21 X11).  One wave and four, us: 100 tokens of 32 heads of 128 12.6
// and 7.2, 300 of 48 13.6 and 8.4, 1024 of 32 16.2 and 12.5 (33 MB in and out), 900 of 64 20 and 20.
template <int DK>
__global__ __launch_bounds__(256) void gdn_chunk_kernel(Args a) {
  constexpr int NC = DK / 32;
  constexpr int kKRow = DK + 8;  // 16-bit elements per row of K in LDS
  __shared__ __align__(16) float sA[kChunk * kPitch];  // k_s . k_t, then L, then M'
  __shared__ __align__(16) float sB[kChunk * kPitch];  // k_s . q_t, then Lq
  __shared__ __align__(16) float sX[kChunk * kPitch];  // the two triangles' inverses
  __shared__ __align__(16) uint16_t sK[kChunk * kKRow];
  __shared__ __align__(16) float sGate[kChunk], sBeta[kChunk];
  __shared__ int sFinite[4];

  const int hv = blockIdx.x % a.Hv, rest = blockIdx.x / a.Hv;
  const int chunk = rest % a.chunks, slot = rest / a.chunks;
  const int per = a.Hv / a.Hk, hk = hv / per;
  const bool writes_k = hv % per == 0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  const int t0 = chunk * kChunk;
  const size_t slotT = (size_t)slot * a.T;

  // Rows 16 i + li of K or Q; those of masked and missing tokens are zeros.
  auto load_rows = [&](const uint16_t* from, int i, uint4 (&f)[NC]) __attribute__((always_inline)) {
    int t = t0 + 16 * i + li;
    const bool past = t >= a.T;
    t = past ? a.T - 1 : t;
    const size_t row = ((slotT + t) * a.Hk + hk) * DK + 8 * kq;
    const bool on = !past && (a.mask == nullptr || a.mask[slotT + t] != 0);
#pragma unroll
    for (int C = 0; C < NC; ++C) {
      f[C] = *reinterpret_cast<const uint4*>(from + row + 32 * C);
      if (!on) f[C] = uint4{0u, 0u, 0u, 0u};
    }
  };
  float finite = 0.f;  // stays zero
  // rows s = 16 ts + 4 kq + r, column t = 16 tt + li (with the diagonals k . k and k . q among them: nothing that is not finite in K or Q
  // stays unseen)
  auto product = [&](const uint4 (&left)[NC], const uint4 (&right)[NC], int ts, int tt, float* to) __attribute__((always_inline)) {
    f32x4_t x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int C = 0; C < NC; ++C) x = mfma(left[C], right[C], x);
#pragma unroll
    for (int e = 0; e < 4; ++e) finite = fmaf(x[e], 0.f, finite);
    *reinterpret_cast<f32x4_t*>(to + (16 * tt + li) * kPitch + 16 * ts + 4 * kq) = x;
  };
  uint32_t on_bits = 0;
  {  // (every wave has the bits, the last one the gates)
    const int t = t0 + (lane & 31);
    const bool on = t < a.T && (a.mask == nullptr || a.mask[slotT + t] != 0);
    on_bits = (uint32_t)__ballot(on);
    if (wave == 3) {
      const size_t at = (slotT + (t < a.T ? t : a.T - 1)) * a.Hv + hv;
      float g = load_as_f32(a.g, at, a.g_dtype), beta = load_as_f32(a.beta, at, a.beta_dtype);
      g = on ? g : 1.f, beta = on ? beta : 0.f;
      if (lane < kChunk) sGate[lane] = g, sBeta[lane] = beta;
      finite = fmaf(g, 0.f, beta * 0.f);
    }
  }
  {
    uint4 f0[NC], f1[NC], f2[NC];
    if (wave == 0) {
      load_rows(a.k, 0, f0), load_rows(a.k, 1, f1);
      product(f0, f0, 0, 0, sA), product(f0, f1, 0, 1, sA);
    } else if (wave == 1) {
      load_rows(a.k, 1, f0), load_rows(a.q, 1, f1);
      product(f0, f0, 1, 1, sA), product(f0, f1, 1, 1, sB);
    } else if (wave == 2) {
      load_rows(a.k, 0, f0), load_rows(a.q, 0, f1), load_rows(a.q, 1, f2);
      product(f0, f1, 0, 0, sB), product(f0, f2, 0, 1, sB);
    } else if (writes_k) {
      load_rows(a.k, 0, f0), load_rows(a.k, 1, f1);
#pragma unroll
      for (int C = 0; C < NC; ++C) {
        *reinterpret_cast<uint4*>(sK + li * kKRow + 32 * C + 8 * kq) = f0[C];
        *reinterpret_cast<uint4*>(sK + (16 + li) * kKRow + 32 * C + 8 * kq) = f1[C];
      }
    }
  }
  __syncthreads();
  const size_t here = ((size_t)slot * a.chunks + chunk) * chunk_bytes<DK>(a);
  char* const out = a.work + here + (size_t)hv * kHeadBytes;
  float* const vec = reinterpret_cast<float*>(out + 2 * kMatBytes);
  if (wave < 2) {
    // one column s per lane: the lower half of the wave L, the upper half Lq; tokens 16 wave .. + 15
    const int s = lane & 31;
    const bool lower = lane < 32;
    float* const mat = (lower ? sA : sB) + s;
    f32x4_t gate[kChunk / 4], beta[4];
#pragma unroll
    for (int t = 0; t < kChunk / 4; ++t) gate[t] = *reinterpret_cast<const f32x4_t*>(sGate + 4 * t);
#pragma unroll
    for (int t = 0; t < 4; ++t) beta[t] = *reinterpret_cast<const f32x4_t*>(sBeta + 16 * wave + 4 * t);
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) x[t] = mat[(16 * wave + t) * kPitch];
    float r = 0.f, c_mine = 0.f, c = 1.f;
    auto step = [&](int t) __attribute__((always_inline)) {
      const float g = gate[t >> 2][t & 3];
      r = t == s ? 1.f : (t > s ? r * g : 0.f);
      c *= g;
      c_mine = t == s ? c : c_mine;
    };
    auto entries = [&](auto half) __attribute__((always_inline)) {
      constexpr int H = decltype(half)::value;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = 16 * H + i;
        step(t);
        const bool counts = lower ? t > s : t >= s && ((on_bits >> t) & 1u) != 0;  // (a masked token's y is zero)
        const float entry = counts ? (lower ? beta[i >> 2][i & 3] * r * x[i] : r * x[i]) : 0.f;
        mat[t * kPitch] = entry;
        finite = fmaf(entry, 0.f, finite);
      }
    };
    if (wave == 0) {
      entries(std::integral_constant<int, 0>{});
    } else {
#pragma unroll
      for (int t = 0; t < 16; ++t) step(t);
      entries(std::integral_constant<int, 1>{});
      finite = fmaf(r, 0.f, fmaf(c, 0.f, finite));
      if (lower) {
        vec[s] = ((on_bits >> s) & 1u) != 0 ? c_mine : 0.f;
        vec[kChunk + s] = r;
        if (s == 0) vec[kTail] = c, vec[kTail + 2] = __uint_as_float(on_bits);
      }
    }
  } else if (writes_k) {
    // K^T: lane (li, kq) takes row dk_of(c, li) of tokens token_of(kq, 0 .. 7), four of them by a transposing read: its lane 4 e + q points
    // at token 4 kq + e and four dk, lane t receives element t % 4 of lanes t / 4, 4 + t / 4, 8 + t / 4, 12 + t / 4
    typedef short s16x4_t __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
    char* const kt = a.work + here + (size_t)a.Hv * kHeadBytes + (size_t)hk * (kChunk * DK * 2);
    const uint16_t* const from = sK + (4 * kq + (li >> 2)) * kKRow + 8 * (li & 3);
#pragma unroll
    for (int i = 0; i < DK / 32; ++i) {
      const int c = (wave - 2) * (DK / 32) + i, dk = 32 * (c >> 1) + 4 * (c & 1);
      const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(from + dk)));
      const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(from + 16 * kKRow + dk)));
      reinterpret_cast<uint4*>(kt)[c * 64 + lane] = uint4{lo.x, lo.y, hi.x, hi.y};
    }
  }
  __syncthreads();
  auto store_pieces = [&](const float* mat, int m, int i) __attribute__((always_inline)) {
    const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(mat + (16 * i + li) * kPitch + 4 * kq);
    const f32x4_t hi = *reinterpret_cast<const f32x4_t*>(mat + (16 * i + li) * kPitch + 16 + 4 * kq);
    const float f[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    const Pieces<8> p = split_bf16(f);
    uint4* dst = reinterpret_cast<uint4*>(out + m * kMatBytes + i * 3072) + lane;
    dst[0] = uint4{p.hi[0], p.hi[1], p.hi[2], p.hi[3]};
    dst[64] = uint4{p.mid[0], p.mid[1], p.mid[2], p.mid[3]};
    dst[128] = uint4{p.lo[0], p.lo[1], p.lo[2], p.lo[3]};
  };
  if (wave == 0) {
    // column j of the inverse of either triangle by forward substitution, lanes 0 .. 15 the first, 16 .. 31 the second (the rest as these)
    const int first = lane & 16, j = li;
    float x[16];
    f32x4_t row[2][4];  // the row in use and the next one
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      if (t + 1 < 16) {
#pragma unroll
        for (int s4 = 0; s4 < t + 1; s4 += 4) row[(t + 1) & 1][s4 / 4] = *reinterpret_cast<const f32x4_t*>(sA + (first + t + 1) * kPitch + first + s4);
      }
      float acc0 = t == j ? 1.f : 0.f, acc1 = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) {
        if (s & 1) acc1 -= row[t & 1][s / 4][s & 3] * x[s];
        else acc0 -= row[t & 1][s / 4][s & 3] * x[s];
      }
      x[t] = acc0 + acc1;
      asm volatile("" : "+v"(x[t]));  // row by row
      __builtin_amdgcn_sched_barrier(0);
    }
    if (lane < 32) {
#pragma unroll
      for (int t = 0; t < 16; ++t) sX[(first + t) * kPitch + first + j] = x[t];
    }
    asm volatile("" ::: "memory");  // (one wave: what it has written is there for its reads)
    // k of a product in the order 4 kq + step
    const f32x4_t l21 = *reinterpret_cast<const f32x4_t*>(sA + (16 + li) * kPitch + 4 * kq);
    f32x4_t below = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int step = 0; step < 4; ++step) below = mfma4(l21[step], sX[(4 * kq + step) * kPitch + li], below);
    const f32x4_t x22 = *reinterpret_cast<const f32x4_t*>(sX + (16 + li) * kPitch + 16 + 4 * kq);
    f32x4_t x21 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int step = 0; step < 4; ++step) x21 = mfma4(x22[step], below[step], x21);
    const float beta = sBeta[first + j], beta0 = sBeta[li];
    if (lane < 32) {
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const float m = x[t] * beta;
        finite = fmaf(m, 0.f, finite);
        sA[(first + t) * kPitch + first + j] = m;  // (above the triangles L's zeros stay)
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float m = -x21[e] * beta0;
      finite = fmaf(m, 0.f, finite);
      sA[(16 + 4 * kq + e) * kPitch + li] = m;
    }
  } else if (wave >= 2) {
    store_pieces(sB, 1, wave - 2);
  }
  {
    const bool all_finite = __all(finite == 0.f);
    if (lane == 0) sFinite[wave] = all_finite;
  }
  __syncthreads();
  if (wave < 2) store_pieces(sA, 0, wave);
  if (threadIdx.x == 64) vec[kTail + 1] = sFinite[0] & sFinite[1] & sFinite[2] & sFinite[3] ? 0.f : __builtin_nanf("");
}

// MASKED: some tokens may not count (those past T read zeros and need no looking after).  WAVES: of a workgroup, which
// divide the DK elements of a row among themselves, 1 or DK / 32.
template <int DK, bool MASKED, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(1, WAVES == 1 ? 1 : 2)))
void gdn_prompt_kernel(Args a) {
  constexpr int NC = DK / 32 / WAVES, NT = 2 * NC;  // pieces of 32 and of 16 dk that a wave has
  constexpr int kTiles = WAVES == 1 ? 2 : 1;         // of the tokens whose Y it computes
  constexpr bool kEarly = WAVES > 1;                 // c and c_T / c_s of the next chunk are asked for at their last use, not last
  constexpr int kStored = WAVES == 4 ? 2 : 4;        // tokens of a lane's four there whose results it writes
  // the waves' parts of U (two tiles) and W, those of a chunk while the ones before may still be read
  __shared__ f32x4_t parts[2][WAVES][4][WAVES == 1 ? 1 : 64];
  __shared__ float sums[WAVES][16];  // (token by token: their parts of one row each)
  const int slices = a.Dv / 16;
  // the slices of a head read the same K, Q, M' and Lq: all of them behind one L2 (blocks go to the XCDs in turn)
  const int heads = a.slots * a.Hv;
  int item, slice;
  if (heads % 8 == 0) {
    const int b = blockIdx.x / 8;
    item = (b / slices) * 8 + blockIdx.x % 8;
    slice = b % slices;
  } else {
    item = blockIdx.x / slices;
    slice = blockIdx.x % slices;
  }
  const int slot = item / a.Hv, hv = item % a.Hv, hk = hv / (a.Hv / a.Hk);
  const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
  const int wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile0 = WAVES == 4 ? wave >> 1 : wave;          // the first (or only) tile of tokens whose Y it computes
  const int first = WAVES == 4 ? 2 * (wave & 1) : 0;        // of a lane's four tokens there
  const size_t slotT = (size_t)slot * a.T;
  const int dv = 16 * slice + li;

  // S^T tile c of this wave: rows dk_of(NT wave + c, 4 kq + r), column dv = this lane's; two tiles are 8 consecutive dk of a
  // row of S
  f32x4_t st[NT];
  const size_t srow = ((size_t)item * a.Dv + dv) * DK + 32 * NC * wave + 8 * kq;
#pragma unroll
  for (int C = 0; C < NC; ++C)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (a.state_in == nullptr) {
        st[2 * C + h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      } else if (a.state_dtype == DFLASH_FP32) {
        st[2 * C + h] = *reinterpret_cast<const f32x4_t*>((const float*)a.state_in + srow + 32 * C + 4 * h);
      } else {
        const uint2 w = *reinterpret_cast<const uint2*>((const uint16_t*)a.state_in + srow + 32 * C + 4 * h);
        const uint32_t b[4] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16};
#pragma unroll
        for (int e = 0; e < 4; ++e) st[2 * C + h][e] = a.state_dtype == DFLASH_BF16 ? bf16_bits_to_f32(b[e]) : f16_bits_to_f32(b[e]);
      }
    }

  // What a chunk reads and writes by token goes through buffer descriptors of this slot: tokens past T read
  // zeros and are not written, with no branch (a branch around a store leaves the count of requests in flight
  // open, and the next wait for a load becomes a wait for every store).
  const uint32_t k_bytes = (uint32_t)a.T * a.Hk * DK * 2, v_bytes = (uint32_t)a.T * a.Hv * a.Dv * 2;
  const auto k_buf = buffer_of(a.k + slotT * a.Hk * DK, k_bytes), q_buf = buffer_of(a.q + slotT * a.Hk * DK, k_bytes);
  const auto v_buf = buffer_of(a.v + slotT * a.Hv * a.Dv, v_bytes), y_buf = buffer_of(a.y + slotT * a.Hv * a.Dv, v_bytes);
  const auto tape_buf = buffer_of(a.tape + slotT * a.Hv * a.Dv, a.tape != nullptr ? 2 * v_bytes : 0u);
  const uint32_t k_step = (uint32_t)a.Hk * DK * 2, v_step = (uint32_t)a.Hv * a.Dv * 2;  // bytes per token
  const uint32_t k_at = li * k_step + hk * (DK * 2) + 64 * NC * wave + 16 * kq;
  const uint32_t v_at = 4 * kq * v_step + (hv * a.Dv + dv) * 2;

  uint4 kf[2][NC], qf[2][NC], kt[NT], mf[2][3], lf[kTiles][3];
  uint32_t vb[8];
  f32x4_t cv[2], cfv[2];
  f32x4_t tail_next;  // (asked for with K and Q: the scheduler moves the scaling of S to the front)
  const size_t per_chunk = chunk_bytes<DK>(a);
  const char* const head0 = a.work + (size_t)slot * a.chunks * per_chunk + (size_t)hv * kHeadBytes;
  const char* const kt0 = a.work + (size_t)slot * a.chunks * per_chunk + (size_t)a.Hv * kHeadBytes + (size_t)hk * (kChunk * DK * 2);
  auto load_kq = [&](int ch) __attribute__((always_inline)) {
    tail_next = reinterpret_cast<const f32x4_t*>(head0 + ch * per_chunk + 2 * kMatBytes + 4 * kTail)[lane >> 6];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t at = k_at + (ch * kChunk + 16 * i) * k_step;
#pragma unroll
      for (int C = 0; C < NC; ++C) {
        kf[i][C] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(k_buf, at + 64 * C, 0, 0));
        qf[i][C] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(q_buf, at + 64 * C, 0, 0));
      }
    }
  };
  auto load_v = [&](int ch) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      vb[j] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(v_buf, v_at + (ch * kChunk + 16 * (j >> 2) + (j & 3)) * v_step, 0, 0);
  };
  auto load_m = [&](int ch) __attribute__((always_inline)) {
    const uint4* src = reinterpret_cast<const uint4*>(head0 + ch * per_chunk) + lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) mf[i][p] = src[(3 * i + p) * 64];
  };
  auto load_l = [&](int ch) __attribute__((always_inline)) {
    const uint4* src = reinterpret_cast<const uint4*>(head0 + ch * per_chunk + kMatBytes) + 3 * tile0 * 64 + lane;
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) lf[i][p] = src[(3 * i + p) * 64];
  };
  auto load_kt = [&](int ch) __attribute__((always_inline)) {
    const uint4* src = reinterpret_cast<const uint4*>(kt0 + ch * per_chunk) + NT * wave * 64 + lane;
#pragma unroll
    for (int c = 0; c < NT; ++c) kt[c] = src[c * 64];
  };
  auto load_vec = [&](int ch, int which, f32x4_t (&f)[2]) __attribute__((always_inline)) {
    const float* vec = reinterpret_cast<const float*>(head0 + ch * per_chunk + 2 * kMatBytes) + which * kChunk;
#pragma unroll
    for (int i = 0; i < 2; ++i) f[i] = *reinterpret_cast<const f32x4_t*>(vec + 16 * i + 4 * kq);
  };
  // arithmetic may move across, requests to memory stay where they were written
#define DFLASH_KEEP_REQUESTS() __builtin_amdgcn_sched_barrier(0xF)
  // a barrier for what the waves hand over through LDS; requests to memory stay in flight
  auto meet = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  // sum of the six piece products of two fp32 factors that matter; two accumulators, smaller terms first
  auto product6 = [&](const uint4 (&f)[3], const Pieces<8>& p, f32x4_t big) __attribute__((always_inline)) {
    f32x4_t small = {0.f, 0.f, 0.f, 0.f};
    small = mfma(f[0], p.lo, small);
    big = mfma(f[0], p.mid, big);
    small = mfma(f[2], p.hi, small);
    big = mfma(f[1], p.hi, big);
    small = mfma(f[1], p.mid, small);
    big = mfma(f[0], p.hi, big);
    return big + small;
  };
  // sum over all waves of what each has for the lane's row of S, in the order of the waves
  auto over_waves = [&](float x) __attribute__((always_inline)) -> float {
    x += __shfl_xor(x, 16, 64);
    x += __shfl_xor(x, 32, 64);
    if (WAVES == 1) return x;
    if (kq == 0) sums[wave][li] = x;
    meet();
    float sum = sums[0][li];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += sums[w][li];
    meet();
    return sum;
  };

  // The recurrence itself, for a chunk with numbers that are not finite.
  auto token_by_token = [&](int ch) __attribute__((always_inline)) {
    const int end = (ch + 1) * kChunk < a.T ? (ch + 1) * kChunk : a.T;
#pragma unroll 1
    for (int t = ch * kChunk; t < end; ++t) {
      const uint32_t at = (uint32_t)t * v_step + (hv * a.Dv + dv) * 2;
      float delta = 0.f, y = 0.f;
      if (a.mask == nullptr || a.mask[slotT + t] != 0) {
        const float g = load_as_f32(a.g, (slotT + t) * a.Hv + hv, a.g_dtype);
        const float beta = load_as_f32(a.beta, (slotT + t) * a.Hv + hv, a.beta_dtype);
        const float v = bf16_bits_to_f32((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(v_buf, at, 0, 0));
        const size_t row = ((slotT + t) * a.Hk + hk) * DK + 32 * NC * wave + 8 * kq;
        auto element = [](uint4 w, int e) __attribute__((always_inline)) {  // 0 .. 7
          const uint32_t half[4] = {w.x, w.y, w.z, w.w};
          return __uint_as_float(e & 1 ? half[e >> 1] & 0xffff0000u : half[e >> 1] << 16);
        };
        uint4 kw[NC], qw[NC];
#pragma unroll
        for (int C = 0; C < NC; ++C) {
          kw[C] = *reinterpret_cast<const uint4*>(a.k + row + 32 * C);
          qw[C] = *reinterpret_cast<const uint4*>(a.q + row + 32 * C);
        }
        float known = 0.f;  // S k, summed over the four lanes of every wave that hold a row of S
#pragma unroll
        for (int C = 0; C < NC; ++C)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            f32x4_t& entry = st[2 * C + (e >> 2)];
            entry[e & 3] *= g;
            known = fmaf(entry[e & 3], element(kw[C], e), known);
          }
        delta = (v - over_waves(known)) * beta;
#pragma unroll
        for (int C = 0; C < NC; ++C)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            f32x4_t& entry = st[2 * C + (e >> 2)];
            entry[e & 3] = fmaf(element(kw[C], e), delta, entry[e & 3]);
            y = fmaf(entry[e & 3], element(qw[C], e), y);
          }
        y = over_waves(y);
      }
      if (kq == 0 && wave == 0) {
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (__bf16)y), y_buf, at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(delta), tape_buf, 2 * at, 0, 0);
      }
    }
  };

  // (the way to the token-by-token form leaves the loop: the loop itself stays without a branch around its stores.  Every
  // wave leaves it at the same chunk: what they look at, Delta, is the same numbers in all of them.)
  int ch = 0;
  while (ch < a.chunks) {
    load_kq(ch);
    DFLASH_KEEP_REQUESTS();  // in the order of the loop: what its first wait may leave in flight is the least of both
    load_v(ch);
    if (kEarly) load_vec(ch, 0, cv);
    load_m(ch);
    if (kEarly) load_vec(ch, 1, cfv);
    load_kt(ch);
    load_l(ch);
    if (!kEarly) load_vec(ch, 0, cv), load_vec(ch, 1, cfv);
    DFLASH_KEEP_REQUESTS();
#pragma unroll 1
    for (; ch < a.chunks; ++ch) {
      const int next = ch + 1 < a.chunks ? ch + 1 : ch;
      const float c_last = tail_next[0];
      float finite = tail_next[1];  // stays zero
      const uint32_t on_bits = __float_as_uint(tail_next[2]);
      // ---- U = K S^T, W = Q S^T: rows = tokens, column = dv ---------------------------------------
      f32x4_t U[2], W[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) U[i] = W[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int C = 0; C < NC; ++C) {
        const float f[8] = {st[2 * C][0],     st[2 * C][1],     st[2 * C][2],     st[2 * C][3],
                            st[2 * C + 1][0], st[2 * C + 1][1], st[2 * C + 1][2], st[2 * C + 1][3]};
        const Pieces<8> sp = split_bf16(f);
#pragma unroll
        for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][C], sp.lo, U[i]), W[i] = mfma(qf[i][C], sp.lo, W[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][C], sp.mid, U[i]), W[i] = mfma(qf[i][C], sp.mid, W[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][C], sp.hi, U[i]), W[i] = mfma(qf[i][C], sp.hi, W[i]);
      }
      if constexpr (WAVES > 1) {  // the sums over the waves, in their order: the same numbers in every wave
#pragma unroll
        for (int i = 0; i < 2; ++i) parts[ch & 1][wave][i][lane] = U[i], parts[ch & 1][wave][2 + i][lane] = W[i];
      }
      load_kq(next);
      DFLASH_KEEP_REQUESTS();
      if constexpr (WAVES > 1) {
        meet();
        auto total = [&](int part) __attribute__((always_inline)) -> f32x4_t {
          f32x4_t sum = parts[ch & 1][0][part][lane];
#pragma unroll
          for (int w = 1; w < WAVES; ++w) sum += parts[ch & 1][w][part][lane];
          return sum;
        };
        U[0] = total(0), U[1] = total(1), W[0] = total(2 + tile0);
      }
      // ---- Delta = M' (V - c U) ----------------------------------------------------------------------
      float rhs[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        rhs[j] = bf16_bits_to_f32(vb[j]) - cv[j >> 2][j & 3] * U[j >> 2][j & 3];
        if (MASKED) rhs[j] = __int_as_float(__float_as_int(rhs[j]) & -(int)((on_bits >> token_of(kq, j)) & 1u));
      }
      if (kEarly) W[0] *= tile0 ? cv[1] : cv[0];
      load_v(next);
      if (kEarly) load_vec(next, 0, cv);
      DFLASH_KEEP_REQUESTS();
      const Pieces<8> rp = split_bf16(rhs);
      f32x4_t D[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) D[i] = product6(mf[i], rp, f32x4_t{0.f, 0.f, 0.f, 0.f});
      load_m(next);
      DFLASH_KEEP_REQUESTS();
      // a number that is not finite in V, U (and so in S) or M' is one in every Delta of its column
#pragma unroll
      for (int j = 0; j < 8; ++j) finite = fmaf(D[j >> 2][j & 3], 0.f, finite);
      if (!__all(finite == 0.f)) break;
      // ---- S^T = c_T S^T + K^T diag(c_T / c_s) Delta ----------------------------------------------
      float scaled[8], plain[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        plain[j] = D[j >> 2][j & 3];
        scaled[j] = plain[j] * cfv[j >> 2][j & 3];
      }
      if (kEarly) {
        load_vec(next, 1, cfv);
        DFLASH_KEEP_REQUESTS();
      }
      {
        const Pieces<8> dp = split_bf16(scaled);
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] *= c_last;
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] = mfma(kt[c], dp.lo, st[c]);
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] = mfma(kt[c], dp.mid, st[c]);
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] = mfma(kt[c], dp.hi, st[c]);
      }
      load_kt(next);
      DFLASH_KEEP_REQUESTS();
      // ---- Y = c W + Lq Delta, for the tokens of this wave's tiles -------------------------------------
      const Pieces<8> dq = split_bf16(plain);
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
        const f32x4_t Y = product6(lf[i], dq, kEarly ? W[i] : W[i] * cv[i]), mine = i == 1 || (WAVES > 1 && tile0) ? D[1] : D[0];
#pragma unroll
        for (int r = 0; r < kStored; ++r) {
          const float y_r = kStored == 2 && first ? Y[(r + 2) & 3] : Y[r], d_r = kStored == 2 && first ? mine[(r + 2) & 3] : mine[r];
          const int t = 16 * (tile0 + i) + first + r;  // and 4 kq, which v_at holds
          const uint32_t at = v_at + (ch * kChunk + t) * v_step;
          uint16_t y = __builtin_bit_cast(uint16_t, (__bf16)y_r);
          if (MASKED) y &= (uint16_t)-(int)((on_bits >> (t + 4 * kq)) & 1u);
          __builtin_amdgcn_raw_buffer_store_b16(y, y_buf, at, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(d_r), tape_buf, 2 * at, 0, 0);
        }
      }
      load_l(next);
      if (!kEarly) load_vec(next, 0, cv), load_vec(next, 1, cfv);
      DFLASH_KEEP_REQUESTS();
    }
    if (ch < a.chunks) token_by_token(ch++);
  }
#undef DFLASH_KEEP_REQUESTS

#pragma unroll
  for (int C = 0; C < NC; ++C)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4_t entry = st[2 * C + h];
      if (a.state_dtype == DFLASH_FP32) {
        *reinterpret_cast<f32x4_t*>((float*)a.state_out + srow + 32 * C + 4 * h) = entry;
      } else {
        uint32_t b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = a.state_dtype == DFLASH_BF16 ? f32_to_bf16_bits(entry[e]) : f32_to_f16_bits(entry[e]);
        *reinterpret_cast<uint2*>((uint16_t*)a.state_out + srow + 32 * C + 4 * h) = uint2{b[0] | (b[1] << 16), b[2] | (b[3] << 16)};
      }
    }
}

template <int DK>
int launch(const Args& a, hipStream_t s) {
  hipLaunchKernelGGL((gdn_chunk_kernel<DK>), dim3((unsigned)(a.slots * a.chunks * a.Hv)), dim3(256), 0, s, a);
  const int groups = a.slots * a.Hv * (a.Dv / 16);
  const bool spread = groups <= kSpread;
  const void* fn = a.mask != nullptr ? (spread ? (const void*)gdn_prompt_kernel<DK, true, DK / 32> : (const void*)gdn_prompt_kernel<DK, true, 1>)
                                     : (spread ? (const void*)gdn_prompt_kernel<DK, false, DK / 32> : (const void*)gdn_prompt_kernel<DK, false, 1>);
  Args args = a;
  void* argv[] = {&args};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)groups), dim3(spread ? 2 * DK : 64), argv, 0, s));
  DFLASH_HIP_OK(hipGetLastError());
  return DFLASH_OK;
}

}  // namespace prompt

// Blocks of up to 16 tokens have kernels of their own (one launch, one wave of workgroups per head).
bool gdn_prompt_covers(int slots, int T, int Hk, int Hv, int Dk, int Dv, int in_dtype, int g_per_dk) {
  return in_dtype == DFLASH_BF16 && !g_per_dk && T > 16 && (Dk == 64 || Dk == 128) && Dv % 16 == 0 && Hk > 0 && Hv % Hk == 0 &&
         slots > 0 && (long long)slots * Hv * ((T + 31) / 32) < (1ll << 31) && (long long)slots * Hv * (Dv / 16) < (1ll << 31) &&
         ((long long)T + 32) * Hv * Dv * 4 < (1ll << 31) && ((long long)T + 32) * Hk * Dk * 2 < (1ll << 31);  // (buffer offsets)
}

size_t gdn_prompt_workspace_bytes(int slots, int T, int Hk, int Hv, int Dk) {
  const int chunks = (T + prompt::kChunk - 1) / prompt::kChunk;
  return (size_t)slots * chunks * ((size_t)Hv * prompt::kHeadBytes + (size_t)Hk * (prompt::kChunk * Dk * 2));
}

int gdn_prompt_launch(const void* q, const void* k, const void* v, const void* g, const void* beta, const void* state_in,
                      void* state_out, void* y, float* tape, const uint8_t* mask, void* workspace, int slots, int T, int Hk,
                      int Hv, int Dk, int Dv, int g_dtype, int beta_dtype, int state_dtype, hipStream_t s) {
  prompt::Args a;
  a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v; a.g = g; a.beta = beta;
  a.state_in = state_in; a.state_out = state_out; a.y = (uint16_t*)y; a.tape = tape; a.mask = mask;
  a.work = (char*)workspace;
  a.slots = slots; a.T = T; a.chunks = (T + prompt::kChunk - 1) / prompt::kChunk;
  a.Hk = Hk; a.Hv = Hv; a.Dv = Dv;
  a.g_dtype = g_dtype; a.beta_dtype = beta_dtype; a.state_dtype = state_dtype;
  return Dk == 64 ? prompt::launch<64>(a, s) : prompt::launch<128>(a, s);
}
}  // namespace dflash
