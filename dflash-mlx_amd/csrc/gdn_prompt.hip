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
//    32ths (gdn_prompt_spread_kernel): each cuts its part of S into pieces, multiplies and updates it, and the parts of U meet in LDS,
//    one barrier per chunk.  Delta is computed by all of them, from the same sums in the same order.  Four more waves do what the
//    chain does not wait for: two the results, two bring the next chunk's operands.
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
// Measured, 1024 tokens of 32 heads of 128 x 128: 12.5 + 42 us, against 123.7 ms with one workgroup per head that kept S in memory (the
// step-by-step kernel held 41 tokens at most); 600 tokens of 16 heads 7.9 + 23.6.  What the second kernel is bound by is its chain.
// Four waves that did everything took 2950 cycles a chunk (56 and 32 us): a third of them waited for the path to memory, which
// took 124 requests a chunk, M' and vectors for every wave and V two bytes at a time.  Now the chain asks for K and K^T, V is one request
// and a transposing read, the tape's stores are there for those who want it, and a chunk takes 2200 cycles, shared by the
// path through LDS (1000 of them), 160 vector and 18 matrix instructions a wave, and results that the next instruction waits for.
// One wave, 900 tokens of 64 heads: 72 -> 64 us with V and the tape's stores so.  Chunks of
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
// are shared, and what the waves of a row do twice (Delta, the pieces of it) costs more than their chain is shorter: us, one wave and
// several, 300 tokens of 48 heads of 128 x 128 25.2 and 28.5, 900 tokens of 64 64.4 and 74.5.
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

// arithmetic may move across, requests to memory stay where they were written
#define DFLASH_KEEP_REQUESTS() __builtin_amdgcn_sched_barrier(0xF)

// What a workgroup walks: 16 rows of the state of one head, and the addresses of what their chunks read and write.  What a chunk reads
// and writes by token goes through buffer descriptors of this slot: tokens past T read zeros and are not written, with no branch
// (a branch around a store leaves the count of requests in flight open, and the next wait for a load becomes a wait for every store).
template <int DK>
struct Rows {
  const Args& a;
  int item, slice, slot, hv, hk, lane, li, kq, dv;
  size_t slotT, per_chunk;
  __amdgpu_buffer_rsrc_t k_buf, q_buf, v_buf, y_buf, tape_buf;
  uint32_t k_step, v_step;  // bytes per token
  uint32_t k_at, v_at;      // of row li and 16-byte piece kq of K and Q, of token 4 kq and column dv of V
  const char *head0, *kt0;

  __device__ __forceinline__ explicit Rows(const Args& args) : a(args) {
    const int slices = a.Dv / 16;
    // the slices of a head read the same K, Q, M' and Lq: all of them behind one L2 (blocks go to the XCDs in turn)
    const int heads = a.slots * a.Hv;
    if (heads % 8 == 0) {
      const int b = blockIdx.x / 8;
      item = (b / slices) * 8 + blockIdx.x % 8;
      slice = b % slices;
    } else {
      item = blockIdx.x / slices;
      slice = blockIdx.x % slices;
    }
    slot = item / a.Hv, hv = item % a.Hv, hk = hv / (a.Hv / a.Hk);
    lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
    dv = 16 * slice + li;
    slotT = (size_t)slot * a.T;
    const uint32_t k_bytes = (uint32_t)a.T * a.Hk * DK * 2, v_bytes = (uint32_t)a.T * a.Hv * a.Dv * 2;
    k_buf = buffer_of(a.k + slotT * a.Hk * DK, k_bytes), q_buf = buffer_of(a.q + slotT * a.Hk * DK, k_bytes);
    v_buf = buffer_of(a.v + slotT * a.Hv * a.Dv, v_bytes), y_buf = buffer_of(a.y + slotT * a.Hv * a.Dv, v_bytes);
    tape_buf = buffer_of(a.tape + slotT * a.Hv * a.Dv, a.tape != nullptr ? 2 * v_bytes : 0u);
    k_step = (uint32_t)a.Hk * DK * 2, v_step = (uint32_t)a.Hv * a.Dv * 2;
    k_at = li * k_step + hk * (DK * 2) + 16 * kq;
    v_at = 4 * kq * v_step + (hv * a.Dv + dv) * 2;
    per_chunk = chunk_bytes<DK>(a);
    head0 = a.work + (size_t)slot * a.chunks * per_chunk + (size_t)hv * kHeadBytes;
    kt0 = a.work + (size_t)slot * a.chunks * per_chunk + (size_t)a.Hv * kHeadBytes + (size_t)hk * (kChunk * DK * 2);
  }

  // Element 8 kq of piece `first` (of 32 dk) of row dv of the state.
  __device__ __forceinline__ size_t state_at(int first) const { return ((size_t)item * a.Dv + dv) * DK + 32 * first + 8 * kq; }
  // S^T tile c: rows dk_of(2 first + c, 4 kq + r), column dv; two tiles are 8 consecutive dk of a row of S.
  template <int NT>
  __device__ __forceinline__ void load_state(int first, f32x4_t (&st)[NT]) const {
    const size_t srow = state_at(first);
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      const size_t at = srow + 32 * (c >> 1) + 4 * (c & 1);
      if (a.state_in == nullptr) {
        st[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      } else if (a.state_dtype == DFLASH_FP32) {
        st[c] = *reinterpret_cast<const f32x4_t*>((const float*)a.state_in + at);
      } else {
        const uint2 w = *reinterpret_cast<const uint2*>((const uint16_t*)a.state_in + at);
        const uint32_t b[4] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16};
#pragma unroll
        for (int e = 0; e < 4; ++e) st[c][e] = a.state_dtype == DFLASH_BF16 ? bf16_bits_to_f32(b[e]) : f16_bits_to_f32(b[e]);
      }
    }
  }
  template <int NT>
  __device__ __forceinline__ void store_state(int first, const f32x4_t (&st)[NT]) const {
    const size_t srow = state_at(first);
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      const size_t at = srow + 32 * (c >> 1) + 4 * (c & 1);
      if (a.state_dtype == DFLASH_FP32) {
        *reinterpret_cast<f32x4_t*>((float*)a.state_out + at) = st[c];
      } else {
        uint32_t b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = a.state_dtype == DFLASH_BF16 ? f32_to_bf16_bits(st[c][e]) : f32_to_f16_bits(st[c][e]);
        *reinterpret_cast<uint2*>((uint16_t*)a.state_out + at) = uint2{b[0] | (b[1] << 16), b[2] | (b[3] << 16)};
      }
    }
  }

  template <int NC>  // pieces first .. first + NC - 1 of rows 16 i + li of K or Q
  __device__ __forceinline__ void load_rows(__amdgpu_buffer_rsrc_t from, int ch, int i, int first, uint4 (&f)[NC]) const {
    const uint32_t at = k_at + 64 * first + (ch * kChunk + 16 * i) * k_step;
#pragma unroll
    for (int C = 0; C < NC; ++C) f[C] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(from, at + 64 * C, 0, 0));
  }
  __device__ __forceinline__ void load_matrix(int ch, int which, int i, uint4 (&f)[3]) const {  // tile i of M' (0) or Lq (1)
    const uint4* src = reinterpret_cast<const uint4*>(head0 + ch * per_chunk + which * kMatBytes) + lane;
#pragma unroll
    for (int p = 0; p < 3; ++p) f[p] = src[(3 * i + p) * 64];
  }
  template <int NT>
  __device__ __forceinline__ void load_kt(int ch, int first, uint4 (&f)[NT]) const {
    const uint4* src = reinterpret_cast<const uint4*>(kt0 + ch * per_chunk) + 2 * first * 64 + lane;
#pragma unroll
    for (int c = 0; c < NT; ++c) f[c] = src[c * 64];
  }
  __device__ __forceinline__ f32x4_t load_vec(int ch, int which, int i) const {  // of the four tokens of tile i: c (0), c_T / c_s (1)
    return *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(head0 + ch * per_chunk + 2 * kMatBytes) + which * kChunk + 16 * i + 4 * kq);
  }
  __device__ __forceinline__ f32x4_t load_tail(int ch) const {
    return reinterpret_cast<const f32x4_t*>(head0 + ch * per_chunk + 2 * kMatBytes + 4 * kTail)[lane >> 6];
  }

  // Of a chunk, 16 bytes per lane: V of these 16 columns, lane l half l % 2 of token l / 2 (of the last one for those past T, which count for
  // nothing), or the vectors and the four words behind them.  One load either way.
  __device__ __forceinline__ uint4 load_columns(int ch, bool vectors) const {
    constexpr int kLast = (kTail + 4) / 4 - 1;
    int t = ch * kChunk + (lane >> 1);
    t = t < a.T ? t : a.T - 1;
    const size_t of_v = (slotT + t) * v_step + (hv * a.Dv + 16 * slice) * 2 + 16 * (lane & 1);
    const size_t of_vectors = ch * per_chunk + 2 * kMatBytes + 16 * (lane < kLast ? lane : kLast);
    return *reinterpret_cast<const uint4*>((vectors ? head0 : (const char*)a.v) + (vectors ? of_vectors : of_v));
  }

  // Brings a chunk into the L2 that the slices of a head share, a line of 128 bytes per lane of two waves per slice: a chunk's time is about that of
  // one trip to memory, and the operands are asked for one chunk ahead.  What comes back is looked at by nobody; see keep().
  __device__ __forceinline__ uint32_t touch(int ch, int wave) const {
    constexpr int kHeadLines = (kHeadBytes + 127) / 128, kRowLines = DK / 64, kLines = kChunk * kRowLines;
    ch = ch < a.chunks ? ch : a.chunks - 1;
    int line = 64 * (2 * slice + wave) + lane;
    const char* from = head0 + ch * per_chunk + 128 * line;
    if (line >= kHeadLines) {
      line -= kHeadLines;
      const bool turned = line < kLines, of_k = line < 2 * kLines, of_q = line < 3 * kLines;
      const int in = line - (turned ? 0 : of_k ? kLines : of_q ? 2 * kLines : 3 * kLines);
      int t = ch * kChunk + in / kRowLines;
      t = t < a.T ? t : a.T - 1;
      const char* const row = (const char*)(of_k ? a.k : a.q) + (slotT + t) * k_step + hk * (DK * 2) + 128 * (in % kRowLines);
      const int v_lines = (a.Dv + 63) / 64;
      int tv = ch * kChunk + in / v_lines;
      tv = tv < a.T ? tv : a.T - 1;
      const char* const v_row = (const char*)a.v + (slotT + tv) * v_step + hv * a.Dv * 2;
      from = turned ? kt0 + ch * per_chunk + 128 * in : of_q ? row : v_row + (128 * (in % v_lines) < 2 * a.Dv ? 128 * (in % v_lines) : 0);
    }
    return *reinterpret_cast<const uint32_t*>(from);
  }
  static __device__ __forceinline__ void keep(uint32_t touched) { asm volatile("" ::"v"(touched)); }

  // y and the tape of token `t` (and 4 kq) of a chunk
  template <bool MASKED, bool TAPE>
  __device__ __forceinline__ void store_token(int ch, int t, float y_t, float delta, uint32_t on_bits, uint32_t nowhere) const {
    const uint32_t at = (v_at + (ch * kChunk + t) * v_step) | nowhere;  // (2^31 or more is behind every row)
    uint16_t y = __builtin_bit_cast(uint16_t, (__bf16)y_t);
    if (MASKED) y &= (uint16_t)-(int)((on_bits >> (t + 4 * kq)) & 1u);
    __builtin_amdgcn_raw_buffer_store_b16(y, y_buf, at, 0, 0);
    if (TAPE) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(delta), tape_buf, 2 * at | nowhere, 0, 0);
  }

  // The recurrence itself, for a chunk with numbers that are not finite: by one wave, which has all of its rows.
  __device__ __forceinline__ void token_by_token(int ch, f32x4_t (&st)[DK / 16]) const {
    constexpr int NC = DK / 32;
    const int end = (ch + 1) * kChunk < a.T ? (ch + 1) * kChunk : a.T;
    auto over_row = [](float x) __attribute__((always_inline)) {  // the four lanes that hold a row
      x += __shfl_xor(x, 16, 64);
      return x + __shfl_xor(x, 32, 64);
    };
#pragma unroll 1
    for (int t = ch * kChunk; t < end; ++t) {
      const uint32_t at = (uint32_t)t * v_step + (hv * a.Dv + dv) * 2;
      float delta = 0.f, y = 0.f;
      if (a.mask == nullptr || a.mask[slotT + t] != 0) {
        const float g = load_as_f32(a.g, (slotT + t) * a.Hv + hv, a.g_dtype);
        const float beta = load_as_f32(a.beta, (slotT + t) * a.Hv + hv, a.beta_dtype);
        const float v = bf16_bits_to_f32((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(v_buf, at, 0, 0));
        const size_t row = ((slotT + t) * a.Hk + hk) * DK + 8 * kq;
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
        float known = 0.f;  // S k
#pragma unroll
        for (int C = 0; C < NC; ++C)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            f32x4_t& entry = st[2 * C + (e >> 2)];
            entry[e & 3] *= g;
            known = fmaf(entry[e & 3], element(kw[C], e), known);
          }
        delta = (v - over_row(known)) * beta;
#pragma unroll
        for (int C = 0; C < NC; ++C)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            f32x4_t& entry = st[2 * C + (e >> 2)];
            entry[e & 3] = fmaf(element(kw[C], e), delta, entry[e & 3]);
            y = fmaf(entry[e & 3], element(qw[C], e), y);
          }
        y = over_row(y);
      }
      if (kq == 0) {
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (__bf16)y), y_buf, at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(delta), tape_buf, 2 * at, 0, 0);
      }
    }
  }
};

// V of a lane's eight tokens out of a chunk's 16 columns in LDS: a transposing read gives the lane its column of four (see the chunk
// kernel).
typedef uint16_t Columns[kChunk][16];
struct Values {
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  s16x4_t lo, hi;
  __device__ __forceinline__ void read(const Columns& from, int li, int kq) {
    typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
    const uint16_t* const at = &from[4 * kq + (li >> 2)][4 * (li & 3)];
    lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
    hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 16 * 16));
  }
  __device__ __forceinline__ float operator[](int j) const { return bf16_bits_to_f32((uint16_t)(j < 4 ? lo[j & 3] : hi[j & 3])); }
};

// sum of the six piece products of two fp32 factors that matter; two accumulators, smaller terms first
__device__ __forceinline__ f32x4_t product6(const uint4 (&f)[3], const Pieces<8>& p, f32x4_t big) {
  f32x4_t small = {0.f, 0.f, 0.f, 0.f};
  small = mfma(f[0], p.lo, small);
  big = mfma(f[0], p.mid, big);
  small = mfma(f[2], p.hi, small);
  big = mfma(f[1], p.hi, big);
  small = mfma(f[1], p.mid, small);
  big = mfma(f[0], p.hi, big);
  return big + small;
}
__device__ __forceinline__ Pieces<8> split_tiles(f32x4_t x, f32x4_t y) {
  const float f[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  return split_bf16(f);
}
// V - c U for the eight tokens of a lane, what a masked token holds left out
template <bool MASKED>
__device__ __forceinline__ Pieces<8> right_side(const Values& v, const f32x4_t (&cv)[2], const f32x4_t (&U)[2], uint32_t on_bits, int kq) {
  float rhs[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    rhs[j] = v[j] - cv[j >> 2][j & 3] * U[j >> 2][j & 3];
    if (MASKED) rhs[j] = __int_as_float(__float_as_int(rhs[j]) & -(int)((on_bits >> token_of(kq, j)) & 1u));
  }
  return split_bf16(rhs);
}

// One wave with all of its 16 rows.  MASKED: some tokens may not count (those past T read zeros and need no looking after).
template <int DK, bool MASKED, bool TAPE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1))) void gdn_prompt_kernel(Args a) {
  constexpr int NC = DK / 32, NT = 2 * NC;  // pieces of 32 and of 16 dk
  __shared__ __align__(16) Columns values;  // V
  const Rows<DK> rows(a);
  f32x4_t st[NT];
  rows.load_state(0, st);
  uint4 kf[2][NC], qf[2][NC], kt[NT], mf[2][3], lf[2][3];
  uint4 columns;
  f32x4_t cv[2], cfv[2];
  f32x4_t tail_next;  // (asked for with K and Q: the scheduler moves the scaling of S to the front)
  auto load_kq = [&](int ch) __attribute__((always_inline)) {
    tail_next = rows.load_tail(ch);
#pragma unroll
    for (int i = 0; i < 2; ++i) rows.load_rows(rows.k_buf, ch, i, 0, kf[i]), rows.load_rows(rows.q_buf, ch, i, 0, qf[i]);
  };
  auto load_matrices = [&](int ch, int which, uint4 (&f)[2][3]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) rows.load_matrix(ch, which, i, f[i]);
  };
  auto load_vecs = [&](int ch) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) cv[i] = rows.load_vec(ch, 0, i), cfv[i] = rows.load_vec(ch, 1, i);
  };

  // (the way to the token-by-token form leaves the loop: the loop itself stays without a branch around its stores)
  int ch = 0;
  while (ch < a.chunks) {
    load_kq(ch);
    DFLASH_KEEP_REQUESTS();  // in the order of the loop: what its first wait may leave in flight is the least of both
    columns = rows.load_columns(ch, false);
    load_matrices(ch, 0, mf);
    rows.load_kt(ch, 0, kt);
    load_matrices(ch, 1, lf);
    load_vecs(ch);
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
        const Pieces<8> sp = split_tiles(st[2 * C], st[2 * C + 1]);
#pragma unroll
        for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][C], sp.lo, U[i]), W[i] = mfma(qf[i][C], sp.lo, W[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][C], sp.mid, U[i]), W[i] = mfma(qf[i][C], sp.mid, W[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][C], sp.hi, U[i]), W[i] = mfma(qf[i][C], sp.hi, W[i]);
      }
      load_kq(next);
      DFLASH_KEEP_REQUESTS();
      // ---- Delta = M' (V - c U) ----------------------------------------------------------------------
      *reinterpret_cast<uint4*>(&values[rows.lane >> 1][8 * (rows.lane & 1)]) = columns;
      asm volatile("" ::: "memory");  // (one wave: what it has written is there for its reads)
      Values v;
      v.read(values, rows.li, rows.kq);
      const Pieces<8> rp = right_side<MASKED>(v, cv, U, on_bits, rows.kq);
      columns = rows.load_columns(next, false);
      DFLASH_KEEP_REQUESTS();
      f32x4_t D[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) D[i] = product6(mf[i], rp, f32x4_t{0.f, 0.f, 0.f, 0.f});
      load_matrices(next, 0, mf);
      DFLASH_KEEP_REQUESTS();
      // a number that is not finite in V, U (and so in S) or M' is one in every Delta of its column
#pragma unroll
      for (int j = 0; j < 8; ++j) finite = fmaf(D[j >> 2][j & 3], 0.f, finite);
      if (!__all(finite == 0.f)) break;
      // ---- S^T = c_T S^T + K^T diag(c_T / c_s) Delta ----------------------------------------------
      {
        const Pieces<8> dp = split_tiles(D[0] * cfv[0], D[1] * cfv[1]);
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] *= c_last;
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] = mfma(kt[c], dp.lo, st[c]);
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] = mfma(kt[c], dp.mid, st[c]);
#pragma unroll
        for (int c = 0; c < NT; ++c) st[c] = mfma(kt[c], dp.hi, st[c]);
      }
      rows.load_kt(next, 0, kt);
      DFLASH_KEEP_REQUESTS();
      // ---- Y = c W + Lq Delta ---------------------------------------------------------------------------
      const Pieces<8> dq = split_tiles(D[0], D[1]);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const f32x4_t Y = product6(lf[i], dq, W[i] * cv[i]);
#pragma unroll
        for (int r = 0; r < 4; ++r) rows.template store_token<MASKED, TAPE>(ch, 16 * i + r, Y[r], D[i][r], on_bits, 0);
      }
      load_matrices(next, 1, lf);
      load_vecs(next);
      DFLASH_KEEP_REQUESTS();
    }
    if (ch < a.chunks) rows.token_by_token(ch++, st);
  }
  rows.store_state(0, st);
}

// A wave for every 32 elements of the rows.  What bounds it is the chain from a chunk's state to the next one's: S is cut into pieces, the
// waves' parts of U meet in LDS (the chunk's one barrier), and all of them compute Delta from the same sums in the same order and their
// part of the next S.  Q S0^T, Lq Delta and the stores are nobody's input: two more waves, a tile of tokens each, find the pieces of S
// and Delta in LDS and do a chunk's while the next one is under way.  Another two bring what all waves of the chain read, M', V and the
// vectors, to LDS, and the lines of later chunks to the L2.
//   barrier of chunk n: its parts of U, pieces of S, M', V and vectors are there, and Delta of chunk n - 1
// A chunk with numbers that are not finite ends in three more: S is in LDS; one wave has walked the chunk token by token; S is out of LDS again.
template <int DK, bool MASKED, bool TAPE>
__global__ __launch_bounds__(64 * (DK / 32 + 4)) __attribute__((amdgpu_waves_per_eu(1, 2))) void gdn_prompt_spread_kernel(Args a) {
  constexpr int kWaves = DK / 32;
  constexpr int kPitchS = DK + 4;
  __shared__ f32x4_t parts[2][kWaves][2][64];
  __shared__ uint4 pieces[2][kWaves][3][64];
  __shared__ f32x4_t deltas[2][2][64];
  __shared__ uint4 matrix[2][2][3][64];              // M'
  __shared__ __align__(16) Columns values[2];        // V
  __shared__ f32x4_t vectors[2][(kTail + 4) / 4];
  __shared__ int walked[2];
  static_assert(sizeof(pieces[0]) >= 16 * kPitchS * sizeof(float), "a chunk's pieces leave room for S");
  const Rows<DK> rows(a);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = rows.lane, kq = rows.kq;
  // what the waves hand over through LDS is there; requests to memory stay in flight
  auto meet = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // Where a chunk turned out not to be finite: the two barriers of its walk, and that of the chunk behind it (or the last one).
  auto sit_out = [&](int ch) __attribute__((always_inline)) {
    if (!__builtin_amdgcn_readfirstlane(walked[ch & 1])) return false;
    meet();
    meet();
    meet();
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): a loop's waits are for the requests of the loop
    return true;
  };
  if (wave >= kWaves + 2) {  // M', V and the vectors, a chunk ahead
    const int half = wave - kWaves - 2;
    uint4 m0, m1, m2, other;
    auto load_shared = [&](int ch) __attribute__((always_inline)) {
      ch = ch < a.chunks ? ch : a.chunks - 1;
      uint4 m[3];
      rows.load_matrix(ch, 0, half, m);
      m0 = m[0], m1 = m[1], m2 = m[2];  // (as an array across the loop they went to memory)
      other = rows.load_columns(ch, half != 0);
    };
    auto store_shared = [&](int ch) __attribute__((always_inline)) {
      matrix[ch & 1][half][0][lane] = m0, matrix[ch & 1][half][1][lane] = m1, matrix[ch & 1][half][2][lane] = m2;
      if (half == 0) *reinterpret_cast<uint4*>(&values[ch & 1][lane >> 1][8 * (lane & 1)]) = other;
      else if (lane < (kTail + 4) / 4) vectors[ch & 1][lane] = __builtin_bit_cast(f32x4_t, other);
    };
    load_shared(0);
    store_shared(0);
    load_shared(1);
    uint32_t touched = rows.touch(2, half);
    Rows<DK>::keep(rows.touch(3, half));
    meet();
    store_shared(1);
    load_shared(2);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    for (int ch = 1;; ++ch) {
      meet();
      sit_out(ch - 1);
      if (ch == a.chunks) return;
      store_shared(ch + 1);  // (behind the last chunk: the last one, which nobody reads)
      load_shared(ch + 2);
      Rows<DK>::keep(touched);
      touched = rows.touch(ch + 4, half);
    }
  }
  if (wave >= kWaves) {
    const int tile = wave - kWaves;
    uint4 qf[kWaves], lf[3];
    f32x4_t c, W;
    uint32_t on_bits;
    // Q S^T: every wave's part as it would add it up, then the waves in their order
    auto times_state = [&](int ch) __attribute__((always_inline)) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        f32x4_t part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 2; p >= 0; --p) part = mfma(qf[w], pieces[ch & 1][w][p][lane], part);
        W = w == 0 ? part : W + part;
      }
      c = vectors[ch & 1][4 * tile + kq];
      on_bits = __float_as_uint(vectors[ch & 1][kTail / 4][2]);
      rows.load_rows(rows.q_buf, ch + 1 < a.chunks ? ch + 1 : ch, tile, 0, qf);
    };
    rows.load_rows(rows.q_buf, 0, tile, 0, qf);
    rows.load_matrix(0, 1, tile, lf);
    meet();
    times_state(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    for (int ch = 1;; ++ch) {
      meet();
      const uint32_t nowhere = sit_out(ch - 1) ? 0x80000000u : 0u;  // (whose results somebody else has stored)
      const f32x4_t D0 = deltas[(ch - 1) & 1][0][lane], D1 = deltas[(ch - 1) & 1][1][lane], mine = tile ? D1 : D0;
      const f32x4_t Y = product6(lf, split_tiles(D0, D1), W * c);
      rows.load_matrix(ch < a.chunks ? ch : ch - 1, 1, tile, lf);
      DFLASH_KEEP_REQUESTS();
      // (before the stores: a wait for what was asked for behind them is a wait for them)
#pragma unroll
      for (int r = 0; r < 4; ++r) rows.template store_token<MASKED, TAPE>(ch - 1, 16 * tile + r, Y[r], mine[r], on_bits, nowhere);
      if (ch == a.chunks) return;
      DFLASH_KEEP_REQUESTS();
      times_state(ch);
      DFLASH_KEEP_REQUESTS();
    }
  }

  __builtin_amdgcn_s_setprio(2);  // the others have a chunk's time for what they do
  f32x4_t st[2];
  rows.load_state(wave, st);
  uint4 kf[2][1], kt[2];
  auto load_k = [&](int ch) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) rows.load_rows(rows.k_buf, ch, i, wave, kf[i]);
  };
  load_k(0);
  DFLASH_KEEP_REQUESTS();  // in the order of the loop
  rows.load_kt(0, wave, kt);
  DFLASH_KEEP_REQUESTS();
#pragma unroll 1
  for (int ch = 0; ch < a.chunks; ++ch) {
    const int next = ch + 1 < a.chunks ? ch + 1 : ch, now = ch & 1;
    f32x4_t U[2];
    {
      const Pieces<8> sp = split_tiles(st[0], st[1]);
      uint4* const to = &pieces[now][wave][0][lane];
      to[0] = uint4{sp.hi[0], sp.hi[1], sp.hi[2], sp.hi[3]};
      to[64] = uint4{sp.mid[0], sp.mid[1], sp.mid[2], sp.mid[3]};
      to[128] = uint4{sp.lo[0], sp.lo[1], sp.lo[2], sp.lo[3]};
#pragma unroll
      for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][0], sp.lo, f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][0], sp.mid, U[i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) U[i] = mfma(kf[i][0], sp.hi, U[i]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) parts[now][wave][i][lane] = U[i];
    load_k(next);
    DFLASH_KEEP_REQUESTS();
    meet();
    f32x4_t part[2][kWaves], cv[2], cfv[2];
    uint4 mf[2][3];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int w = 0; w < kWaves; ++w) part[i][w] = parts[now][w][i][lane];
    Values v;
    v.read(values[now], rows.li, kq);
#pragma unroll
    for (int i = 0; i < 2; ++i) cv[i] = vectors[now][4 * i + kq];
    const f32x4_t tail = vectors[now][kTail / 4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) mf[i][p] = matrix[now][i][p][lane];
#pragma unroll
    for (int i = 0; i < 2; ++i) cfv[i] = vectors[now][kChunk / 4 + 4 * i + kq];
    __builtin_amdgcn_sched_barrier(0);  // all of them asked for before the first is awaited
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // the sums over the waves, in their order: the same numbers in every wave
      U[i] = part[i][0];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) U[i] += part[i][w];
    }
    const Pieces<8> rp = right_side<MASKED>(v, cv, U, __float_as_uint(tail[2]), kq);
    f32x4_t D[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) D[i] = product6(mf[i], rp, f32x4_t{0.f, 0.f, 0.f, 0.f});
    if (wave < 2) deltas[now][wave][lane] = wave ? D[1] : D[0];
    // a number that is not finite in V, U (and so in S) or M' is one in every Delta of its column; the same in every wave
    float finite = tail[1];  // stays zero
#pragma unroll
    for (int j = 0; j < 8; ++j) finite = fmaf(D[j >> 2][j & 3], 0.f, finite);
    const bool all_finite = __all(finite == 0.f);
    if (wave == 0 && lane == 0) walked[now] = !all_finite;
    if (all_finite) {
      const Pieces<8> dp = split_tiles(D[0] * cfv[0], D[1] * cfv[1]);
#pragma unroll
      for (int c = 0; c < 2; ++c) st[c] = mfma(kt[c], dp.lo, st[c] * tail[0]);
#pragma unroll
      for (int c = 0; c < 2; ++c) st[c] = mfma(kt[c], dp.mid, st[c]);
#pragma unroll
      for (int c = 0; c < 2; ++c) st[c] = mfma(kt[c], dp.hi, st[c]);
    } else {
      // (the pieces of the chunk before are nobody's any more)
      float* const held = reinterpret_cast<float*>(&pieces[now ^ 1][0][0][0]) + rows.li * kPitchS + 8 * kq;
#pragma unroll
      for (int c = 0; c < 2; ++c) *reinterpret_cast<f32x4_t*>(held + 32 * wave + 4 * c) = st[c];
      meet();
      if (wave == 0) {
        f32x4_t all[DK / 16];
#pragma unroll
        for (int c = 0; c < DK / 16; ++c) all[c] = *reinterpret_cast<const f32x4_t*>(held + 32 * (c >> 1) + 4 * (c & 1));
        rows.token_by_token(ch, all);
#pragma unroll
        for (int c = 0; c < DK / 16; ++c) *reinterpret_cast<f32x4_t*>(held + 32 * (c >> 1) + 4 * (c & 1)) = all[c];
      }
      meet();
#pragma unroll
      for (int c = 0; c < 2; ++c) st[c] = *reinterpret_cast<const f32x4_t*>(held + 32 * wave + 4 * c);
      meet();  // (the next chunk's pieces take its place)
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), as above
    }
    rows.load_kt(next, wave, kt);
    DFLASH_KEEP_REQUESTS();
  }
  meet();  // Delta of the last chunk
  rows.store_state(wave, st);
}
#undef DFLASH_KEEP_REQUESTS

template <int DK>
int launch(const Args& a, hipStream_t s) {
  hipLaunchKernelGGL((gdn_chunk_kernel<DK>), dim3((unsigned)(a.slots * a.chunks * a.Hv)), dim3(256), 0, s, a);
  const int groups = a.slots * a.Hv * (a.Dv / 16);
  const bool spread = groups <= kSpread;
  const bool masked = a.mask != nullptr, tape = a.tape != nullptr;
#define DFLASH_PROMPT_FORMS(KERNEL_) \
  (masked ? (tape ? (const void*)KERNEL_<DK, true, true> : (const void*)KERNEL_<DK, true, false>) \
          : (tape ? (const void*)KERNEL_<DK, false, true> : (const void*)KERNEL_<DK, false, false>))
  const void* const fn = spread ? DFLASH_PROMPT_FORMS(gdn_prompt_spread_kernel) : DFLASH_PROMPT_FORMS(gdn_prompt_kernel);
#undef DFLASH_PROMPT_FORMS
  Args args = a;
  void* argv[] = {&args};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)groups), dim3(spread ? 64 * (DK / 32 + 4) : 64), argv, 0, s));
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
