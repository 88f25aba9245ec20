// GatedDeltaNet forward over a block of T tokens that also records the innovation tape,
// for gfx950 (MI355X).
//
// Counterpart of the reference's `gated_delta_tape{,_vec}{,_mask}` Metal kernels
// (dflash_mlx/kernels.py:12-127; array-op form :131-173; dispatcher :176-224): for every
// (batch slot, value head), with the state S[Dv][Dk] (Dk contiguous) and for t = 0..T-1,
//     S      <- g_t * S                      (g_t a scalar per head, or one value per dk)
//     kv     =  S k_t                        (a value per dv)
//     delta  =  (v_t - kv) * beta_t
//     S      <- S + delta (x) k_t
//     y_t    =  S q_t
//     tape_t =  delta                        (fp32)
// and S rounded through the state dtype after every step (kernels.py:96-98; a no-op for an
// fp32 state).  A step whose mask byte is zero leaves S alone and gives y_t = tape_t = 0.
// The tape, with k and g, is what dflash_tape_replay needs to rebuild the state after any
// prefix of the block.
//
// Like the replay, the operation moves the state once in and once out and little else, but
// it is sequential in t, needs two reductions over dk per step, and at 16 steps its
// arithmetic costs about as much as its memory traffic.  Layout for 128 x 128 heads: one
// workgroup of 4 waves per (slot, head); a lane owns 4 rows x 16 columns of S (rows
// 32*wave + 4*(lane/8) + i; columns 4*(lane%8) + 32*c + {0..3}, c = 0..3), so that
//  * a row of S is spread over 8 neighbouring lanes: a reduction over dk is three DPP steps,
//    every lane ends up with the sums and nothing goes through LDS;
//  * every wave load or store of S is eight runs of 128 contiguous bytes;
//  * y_t = (g S) q + (k . q) delta, so one pass over S yields both sums of a step and one
//    reduction round serves both;
//  * with one gate per head and an fp32 state the decay is not applied to S at all: the
//    kernel keeps S / c with c = prod g, scales the two sums and delta instead, and
//    multiplies c back in once at the end (renormalising if c gets very small).
// q, k, v, g, beta of the block are staged once in LDS as fp32.
#include "gdn_device.h"
#include "gdn_block_device.h"
#include <cstdlib>

namespace dflash {
int qmm_stream_grid();  // compute units
namespace {

constexpr int kThreads = 256;

struct GdnArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* g;
  const void* beta;
  const void* state_in;
  void* state_out;
  void* y;
  float* tape;
  const uint8_t* mask;
  int T, Hk, Hv, Dk, Dv;
  Divisor heads, group, row_parts;  // by Hv, by Hv / Hk, by the workgroups of a head (gdn_forward_rows)
  int in_dtype, g_dtype, beta_dtype, state_dtype, g_per_dk;
  int staged;  // step-by-step kernel: steps staged in LDS at a time
  // gated output norm fused behind the recurrence (block kernel only): y is then
  // silu(z) * rms_norm(recurrence output, norm_weight)
  const void* z;  // [slots, T, Hv, Dv], slots and steps with a stride (elements)
  long long z_batch, z_row;
  const void* norm_weight;  // [Dv]
  int weight_dtype;
  float eps;
  BlockArgs block;  // kernels with BLOCK: the block's projections, in place of q, k, v, g and beta
};

// v + (v of the lane the DPP control names): butterfly steps inside a row of 16 lanes -
// quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror (lanes of an aligned group of 8),
// row_mirror (the two groups of 8).
template <int CTRL>
__device__ __forceinline__ float add_dpp(float v) {
  const int o = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true);
  return v + __int_as_float(o);
}
__device__ __forceinline__ float sum_over_8(float v) {
  v = add_dpp<0xB1>(v);
  v = add_dpp<0x4E>(v);
  v = add_dpp<0x141>(v);
  return v;
}
__device__ __forceinline__ float sum_over_16(float v) { return add_dpp<0x140>(sum_over_8(v)); }

__device__ __forceinline__ float dot4(const f32x4_t& s, const float4& k) {
  return s.x * k.x + s.y * k.y + s.z * k.z + s.w * k.w;
}

// ---------------------------------------------------------------------------
// Dk = Dv = 128.  The steps come through LDS in blocks of B = a.staged: (floats) sQ[B][128] |
// sK[B][128] | sV[B][128] | sG[B][128 or 1] | sBeta[B] | sKQ[B].  FOLD: keep S / prod(g) instead of applying the decay (one gate per
// head, fp32 state only).
// ---------------------------------------------------------------------------
template <bool VECG, bool FOLD>
__global__ __launch_bounds__(kThreads) void gdn_forward_128(GdnArgs a) {
  static_assert(!(VECG && FOLD), "the folded decay needs one gate per head");
  extern __shared__ float smem[];
  const int staged = a.staged;
  float* sQ = smem;
  float* sK = sQ + staged * 128;
  float* sV = sK + staged * 128;
  float* sG = sV + staged * 128;
  float* sBeta = sG + staged * (VECG ? 128 : 1);
  float* sKQ = sBeta + staged;

  const int slot = blockIdx.x / a.Hv, hv = blockIdx.x % a.Hv;
  const int hk = hv / (a.Hv / a.Hk);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c3 = lane & 7;
  const int row0 = 32 * wave + 4 * (lane >> 3);  // this lane's rows: row0 .. row0 + 3
  const bool f32_state = FOLD || a.state_dtype == DFLASH_FP32;

  // ---- state in: float4 columns c3 + 8c (c = 0..3) of 4 rows --------------------------------
  const size_t sbase = (size_t)blockIdx.x * 128 * 128;
  f32x4_t st[4][4];
  if (f32_state) {
    const f32x4_t* in = reinterpret_cast<const f32x4_t*>((const float*)a.state_in + sbase);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) st[i][c] = __builtin_nontemporal_load(&in[(row0 + i) * 32 + c3 + 8 * c]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          st[i][c][e] = load_as_f32(a.state_in, sbase + (size_t)(row0 + i) * 128 + 4 * (c3 + 8 * c) + e,
                                    a.state_dtype);
  }

  float cum = 1.f;  // FOLD: the registers hold S / cum
  for (int first = 0; first < a.T; first += staged) {
  const int T = a.T - first < staged ? a.T - first : staged;
  const size_t slotT = (size_t)slot * a.T + first;
  if (first > 0) __syncthreads();  // the block before has been read
  // ---- stage the block ---------------------------------------------------------------------
  for (int i = tid; i < T * 128; i += kThreads) {
    const int t = i >> 7, d = i & 127;
    sQ[i] = load_as_f32(a.q, ((slotT + t) * a.Hk + hk) * 128 + d, a.in_dtype);
    sK[i] = load_as_f32(a.k, ((slotT + t) * a.Hk + hk) * 128 + d, a.in_dtype);
    sV[i] = load_as_f32(a.v, ((slotT + t) * a.Hv + hv) * 128 + d, a.in_dtype);
    if (VECG) sG[i] = load_as_f32(a.g, ((slotT + t) * a.Hv + hv) * 128 + d, a.g_dtype);
  }
  for (int t = tid; t < T; t += kThreads) {
    if (!VECG) sG[t] = load_as_f32(a.g, (slotT + t) * a.Hv + hv, a.g_dtype);
    sBeta[t] = load_as_f32(a.beta, (slotT + t) * a.Hv + hv, a.beta_dtype);
  }
  __syncthreads();
  // k_t . q_t: 16 lanes per step, 8 products each
  for (int t = tid >> 4; t < T; t += kThreads / 16) {
    const int c16 = tid & 15;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) s += sK[t * 128 + 8 * c16 + c] * sQ[t * 128 + 8 * c16 + c];
    s = sum_over_16(s);
    if (c16 == 0) sKQ[t] = s;
  }
  __syncthreads();

  const size_t obase = slotT * a.Hv * 128 + (size_t)hv * 128;  // + t * Hv * 128 + dv
  for (int t = 0; t < T; ++t) {
    float delta[4], yv[4];
    const bool on = a.mask == nullptr || a.mask[slotT + t] != 0;
    if (on) {
      float4 kk[4], qq[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        kk[c] = reinterpret_cast<const float4*>(sK + t * 128)[c3 + 8 * c];
        qq[c] = reinterpret_cast<const float4*>(sQ + t * 128)[c3 + 8 * c];
      }
      const float4 v4 = *reinterpret_cast<const float4*>(sV + t * 128 + row0);
      const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
      const float beta = sBeta[t], kq = sKQ[t];
      if (FOLD) {
        cum *= sG[t];
        if (cum < 1e-12f) {  // same for the whole workgroup: put the scale back into S
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) st[i][c] *= cum;
          cum = 1.f;
        }
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          f32x4_t g4;
          if (VECG) {
            const float4 g = reinterpret_cast<const float4*>(sG + t * 128)[c3 + 8 * c];
            g4 = f32x4_t{g.x, g.y, g.z, g.w};
          } else {
            const float g = sG[t];
            g4 = f32x4_t{g, g, g, g};
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) st[i][c] *= g4;
        }
      }
      float pk[4], pq[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pk[i] = (dot4(st[i][0], kk[0]) + dot4(st[i][1], kk[1])) + (dot4(st[i][2], kk[2]) + dot4(st[i][3], kk[3]));
        pq[i] = (dot4(st[i][0], qq[0]) + dot4(st[i][1], qq[1])) + (dot4(st[i][2], qq[2]) + dot4(st[i][3], qq[3]));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pk[i] = sum_over_8(pk[i]);
        pq[i] = sum_over_8(pq[i]);
      }
      const float rcum = FOLD ? 1.f / cum : 1.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (FOLD) {
          pk[i] *= cum;
          pq[i] *= cum;
        }
        delta[i] = (vv[i] - pk[i]) * beta;
        yv[i] = pq[i] + kq * delta[i];
        const float d = FOLD ? delta[i] * rcum : delta[i];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          st[i][c].x += kk[c].x * d;
          st[i][c].y += kk[c].y * d;
          st[i][c].z += kk[c].z * d;
          st[i][c].w += kk[c].w * d;
        }
      }
      if (!f32_state) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) st[i][c][e] = round_through(st[i][c][e], a.state_dtype);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) delta[i] = 0.f, yv[i] = 0.f;
    }
    // lane c3 = i of each group of 8 lanes writes the outputs of row row0 + i
    float d_out = delta[0], y_out = yv[0];
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      d_out = c3 == i ? delta[i] : d_out;
      y_out = c3 == i ? yv[i] : y_out;
    }
    if (c3 < 4) {
      const size_t o = obase + (size_t)t * a.Hv * 128 + row0 + c3;
      a.tape[o] = d_out;
      store_from_f32(a.y, o, y_out, a.in_dtype);
    }
  }
  }

  // ---- state out ----------------------------------------------------------------------------
  if (f32_state) {
    f32x4_t* out = reinterpret_cast<f32x4_t*>((float*)a.state_out + sbase);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (FOLD) st[i][c] *= cum;
        __builtin_nontemporal_store(st[i][c], &out[(row0 + i) * 32 + c3 + 8 * c]);
      }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          store_from_f32(a.state_out, sbase + (size_t)(row0 + i) * 128 + 4 * (c3 + 8 * c) + e, st[i][c][e],
                         a.state_dtype);
  }
}

// ---------------------------------------------------------------------------
// Dk = 64 or 128, one gate per head, step by step: 16-bit states (which are rounded after every step, so the closed
// form below does not apply) and fp32 states of the head sizes the other kernels do not have.
//  * Rows of S are independent, and a step is a chain (two sums over dk, then the update): what bounds a
//    call of few heads is that chain, so a head is spread over workgroups of 16 R (Dk = 64: 32 R) rows.  A lane
//    holds 8 columns of R rows, a row is 16 (8) neighbouring lanes, its sums are four (three) DPP steps.
//  * k and q of the next step are read from LDS (planes of four, see plane_index) while the present one computes; tape
//    and y leave through LDS, 16 steps at a time.
// Measured against one workgroup per head with 2-byte accesses and the types sorted out per element, bf16 states,
// 16 steps / 1 step, us: 32 heads of 128 x 128 73.9 / 21.7 -> 7.6 / 3.9, 1024 heads 184 / 53 -> 69 / 19; of 64 x 64, whose
// state went through memory at every step, 913 / 77.7 -> 6.8 / 3.4 and 1158 / 105 -> 21 / 5.9.
// ---------------------------------------------------------------------------
template <int STATE, int DK, int R, bool BLOCK>
__global__ __launch_bounds__(kThreads) void gdn_forward_rows(GdnArgs a) {
  constexpr bool kWide = STATE == DFLASH_FP32;
  constexpr int kLanes = DK / 8, kPass = kThreads / kLanes, kRows = kPass * R;  // lanes of a row, rows of a pass, of the workgroup
  constexpr int kD = kRows / 16, kK = DK / 16;  // elements of v and of k, q that a thread brings
  __shared__ __align__(16) float sQ[16 * DK];
  __shared__ __align__(16) float sK[16 * DK];
  __shared__ __align__(16) float sV[16 * kRows];  // v, then (row by row, once it has been read) the tape
  __shared__ __align__(16) float sY[16 * kRows];
  __shared__ __align__(16) float sS[16 * 4];      // gate, beta, k . q of a step
  const int head = a.row_parts.quotient((int)blockIdx.x), row0 = ((int)blockIdx.x - head * (int)a.row_parts.by) * kRows;
  const int slot = a.heads.quotient(head), hv = head - slot * a.Hv, hk = a.group.quotient(hv);
  const int tid = threadIdx.x, t16 = tid >> 4, seg = tid & 15;
  const int rr = tid / kLanes, c8 = tid % kLanes;
  const bool wide = a.in_dtype == DFLASH_FP32;

  const size_t at0 = ((size_t)head * a.Dv + row0 + rr) * DK + 8 * c8;
  u32x4_t raw[R][kWide ? 2 : 1];
  float st[R][8];
  for (int first = 0; first < a.T; first += 16) {
    const int T = a.T - first < 16 ? a.T - first : 16;
    const size_t slotT = (size_t)slot * a.T + first;
    // the block's operands first, the state behind them, nothing looked at before all of it is on its way
    uint32_t rq[kK] = {}, rk[kK] = {}, rv[kD] = {}, g_bits = 0u, beta_bits = 0u;
    // BLOCK: every wave its four steps of q, k and v, of up to four steps in all one of the three; the gates the last wave
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, C = 2 * a.Hk * DK + a.Hv * a.Dv;
    const bool few = T <= 4;
    const int t_b = few ? lane >> 4 : t16, c_q = hk * DK + kK * seg, c_k = c_q + a.Hk * DK, c_v = 2 * a.Hk * DK + hv * a.Dv + row0 + kD * seg;
    auto mine = [&](int which) __attribute__((always_inline)) { return few ? wave == which : 4 * wave < T; };
    ConvRows<kK> b_q, b_k;
    ConvRows<kD> b_v;
    GateBits gates;
    if constexpr (BLOCK) {
      request_rows(a.block, slot, t_b, T, C, c_q, b_q);
      request_rows(a.block, slot, t_b, T, C, c_k, b_k);
      request_rows(a.block, slot, t_b, T, C, c_v, b_v);
      gates = request_gates(a.block, slot, lane < T ? lane : T - 1, hv);
    } else if (t16 < T) {
      load_bits<kK>(a.q, ((slotT + t16) * a.Hk + hk) * DK + kK * seg, wide, rq);
      load_bits<kK>(a.k, ((slotT + t16) * a.Hk + hk) * DK + kK * seg, wide, rk);
      load_bits<kD>(a.v, ((slotT + t16) * a.Hv + hv) * a.Dv + row0 + kD * seg, wide, rv);
    }
    if (!BLOCK && tid < T) {
      const size_t at = (slotT + tid) * a.Hv + hv;
      if (a.g_dtype == DFLASH_FP32) g_bits = ((const uint32_t*)a.g)[at];
      else g_bits = ((const uint16_t*)a.g)[at];
      if (a.beta_dtype == DFLASH_FP32) beta_bits = ((const uint32_t*)a.beta)[at];
      else beta_bits = ((const uint16_t*)a.beta)[at];
    }
    if (first == 0) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const size_t at = at0 + (size_t)i * kPass * DK;
        if (kWide) {
          const u32x4_t* src = reinterpret_cast<const u32x4_t*>((const float*)a.state_in + at);
          raw[i][0] = __builtin_nontemporal_load(src);
          raw[i][kWide ? 1 : 0] = __builtin_nontemporal_load(src + 1);
        } else {
          raw[i][0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>((const uint16_t*)a.state_in + at));
        }
      }
    }
    if constexpr (BLOCK) {
      asm volatile("" ::: "memory");  // every request above is out before the first value is interpreted
      // rows of v are one workgroup's, a key head is kept by the first of its value heads and of its first rows
      const bool keeps = row0 == 0 && hv == hk * (int)a.group.by;
      if (mine(0)) {
        float all[1][kK];
        convolve(a.block, slot, t_b, T, C, c_q, keeps, b_q, all);
        auto& x = all[0];
        normalise<kK, 16>(x, a.block.scale_q, a.block.eps);
#pragma unroll
        for (int e = 0; e < kK; ++e) sQ[t_b * DK + plane_index<DK>(kK * seg + e)] = x[e];
      }
      if (mine(1)) {
        float all[1][kK];
        convolve(a.block, slot, t_b, T, C, c_k, keeps, b_k, all);
        auto& x = all[0];
        normalise<kK, 16>(x, a.block.scale_k, a.block.eps);
#pragma unroll
        for (int e = 0; e < kK; ++e) sK[t_b * DK + plane_index<DK>(kK * seg + e)] = x[e];
        if (keeps && t_b < T && a.block.k_out != nullptr)
          store_exact<kK>(a.block.k_out + ((slotT + t_b) * a.Hk + hk) * DK + kK * seg, x);
      }
      if (mine(2)) {
        float all[1][kD];
        convolve(a.block, slot, t_b, T, C, c_v, true, b_v, all);
        auto& x = all[0];
#pragma unroll
        for (int e = 0; e < kD; ++e) sV[t_b * kRows + kD * seg + e] = x[e];
      }
      if (wave == 3 && lane < T) {
        const float g = gate_of(a.block, gates);
        if (row0 == 0 && a.block.g_out != nullptr) a.block.g_out[(slotT + lane) * a.Hv + hv] = g;
        sS[4 * lane] = g;
        sS[4 * lane + 1] = beta_of(gates);
      }
      __syncthreads();
    } else {
#pragma unroll
      for (int e = 0; e < kK; ++e) asm volatile("" : "+v"(rq[e]), "+v"(rk[e])::"memory");
#pragma unroll
      for (int e = 0; e < kD; ++e) asm volatile("" : "+v"(rv[e])::"memory");
      asm volatile("" : "+v"(g_bits), "+v"(beta_bits)::"memory");
    }
    float kq = 0.f;  // k . q of step t16: 16 lanes, kK products each
#pragma unroll
    for (int e = 0; e < kK; ++e) {
      const int at = t16 * DK + plane_index<DK>(kK * seg + e);
      const float q = BLOCK ? sQ[at] : bits_element(rq, e, a.in_dtype), k = BLOCK ? sK[at] : bits_element(rk, e, a.in_dtype);
      if (!BLOCK) sQ[at] = q, sK[at] = k;
      kq = fmaf(k, q, kq);
    }
    kq = sum_over_16(kq);
    if (seg == 0) sS[4 * t16 + 2] = kq;
    if (!BLOCK) {
#pragma unroll
      for (int e = 0; e < kD; ++e) sV[t16 * kRows + kD * seg + e] = bits_element(rv, e, a.in_dtype);
    }
    if (!BLOCK && tid < 16) {
      const uint32_t g1[1] = {g_bits}, b1[1] = {beta_bits};
      sS[4 * tid] = bits_element(g1, 0, a.g_dtype);
      sS[4 * tid + 1] = bits_element(b1, 0, a.beta_dtype);
    }
    if (first == 0) {
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if constexpr (kWide) st[i][e] = __uint_as_float(raw[i][kWide ? e >> 2 : 0][e & 3]);
          else st[i][e] = e & 1 ? pair_hi<STATE>(raw[i][0][e >> 1]) : pair_lo<STATE>(raw[i][0][e >> 1]);
        }
    }
    __syncthreads();

    f32x4_t k4[2], q4[2], s4;
    float v[R];
    auto fetch = [&](int t) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        k4[h] = *reinterpret_cast<const f32x4_t*>(sK + t * DK + h * (DK / 2) + 4 * c8);
        q4[h] = *reinterpret_cast<const f32x4_t*>(sQ + t * DK + h * (DK / 2) + 4 * c8);
      }
      s4 = *reinterpret_cast<const f32x4_t*>(sS + 4 * t);
#pragma unroll
      for (int i = 0; i < R; ++i) v[i] = sV[t * kRows + i * kPass + rr];
    };
    fetch(0);
    for (int t = 0; t < T; ++t) {
      float kk[8], qq[8], vv[R], delta[R], y[R];
#pragma unroll
      for (int e = 0; e < 8; ++e) kk[e] = k4[e >> 2][e & 3], qq[e] = q4[e >> 2][e & 3];
      const float g = s4[0], beta = s4[1], kdotq = s4[2];
#pragma unroll
      for (int i = 0; i < R; ++i) vv[i] = v[i], delta[i] = y[i] = 0.f;
      fetch(t + 1 < T ? t + 1 : t);
      if (a.mask == nullptr || a.mask[slotT + t] != 0) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
          float pk[2] = {0.f, 0.f}, pq[2] = {0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            st[i][e] *= g;
            pk[e & 1] = fmaf(st[i][e], kk[e], pk[e & 1]);
            pq[e & 1] = fmaf(st[i][e], qq[e], pq[e & 1]);
          }
          const float sk = pk[0] + pk[1], sq = pq[0] + pq[1];
          delta[i] = (vv[i] - (kLanes == 16 ? sum_over_16(sk) : sum_over_8(sk))) * beta;
          y[i] = fmaf(kdotq, delta[i], kLanes == 16 ? sum_over_16(sq) : sum_over_8(sq));
#pragma unroll
          for (int e = 0; e < 8; ++e) st[i][e] = fmaf(kk[e], delta[i], st[i][e]);
          if constexpr (!kWide) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
              const uint32_t w = pack_pair<STATE>(st[i][2 * p], st[i][2 * p + 1]);
              st[i][2 * p] = pair_lo<STATE>(w), st[i][2 * p + 1] = pair_hi<STATE>(w);
            }
          }
        }
      }
      if (c8 == 0) {  // (nobody else reads these elements of v, and this wave has)
#pragma unroll
        for (int i = 0; i < R; ++i) sV[t * kRows + i * kPass + rr] = delta[i], sY[t * kRows + i * kPass + rr] = y[i];
      }
    }
    __syncthreads();
    if (t16 < T) {
      const size_t o = ((slotT + t16) * a.Hv + hv) * a.Dv + row0 + kD * seg;
      float d[kD], y[kD];
#pragma unroll
      for (int e = 0; e < kD; ++e) d[e] = sV[t16 * kRows + kD * seg + e], y[e] = sY[t16 * kRows + kD * seg + e];
      __builtin_memcpy(__builtin_assume_aligned(a.tape + o, kD < 4 ? 4 * kD : 16), d, 4 * kD);
      if (wide) {
        __builtin_memcpy(__builtin_assume_aligned((float*)a.y + o, kD < 4 ? 4 * kD : 16), y, 4 * kD);
      } else {
        uint16_t h[kD];
#pragma unroll
        for (int e = 0; e < kD; ++e) h[e] = (uint16_t)(a.in_dtype == DFLASH_BF16 ? f32_to_bf16_bits(y[e]) : f32_to_f16_bits(y[e]));
        __builtin_memcpy(__builtin_assume_aligned((uint16_t*)a.y + o, kD < 8 ? 2 * kD : 16), h, 2 * kD);
      }
    }
    if (first + 16 < a.T) __syncthreads();  // the next block is staged where this one's results are read
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const size_t at = at0 + (size_t)i * kPass * DK;
    if constexpr (kWide) {
      f32x4_t* dst = reinterpret_cast<f32x4_t*>((float*)a.state_out + at);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        __builtin_nontemporal_store(f32x4_t{st[i][4 * h], st[i][4 * h + 1], st[i][4 * h + 2], st[i][4 * h + 3]}, dst + h);
    } else {
      u32x4_t w;
#pragma unroll
      for (int p = 0; p < 4; ++p) w[p] = pack_pair<STATE>(st[i][2 * p], st[i][2 * p + 1]);  // (exact: rounded already)
      __builtin_nontemporal_store(w, reinterpret_cast<u32x4_t*>((uint16_t*)a.state_out + at));
    }
  }
}

// The form of gdn_forward_rows for a head size and state type; rows: how many a workgroup computes.
template <int STATE, bool BLOCK>
const void* forward_rows_for(int Dk, int Dv, bool many, int* rows) {
  if (Dk == 128 && many && Dv % 32 == 0) return *rows = 32, (const void*)gdn_forward_rows<STATE, 128, 2, BLOCK>;
  if (Dk == 128 && Dv % 16 == 0) return *rows = 16, (const void*)gdn_forward_rows<STATE, 128, 1, BLOCK>;
  if (Dk == 64 && many && Dv % 64 == 0) return *rows = 64, (const void*)gdn_forward_rows<STATE, 64, 2, BLOCK>;
  if (Dk == 64 && Dv % 32 == 0) return *rows = 32, (const void*)gdn_forward_rows<STATE, 64, 1, BLOCK>;
  return nullptr;
}
// Step by step in registers.  Two rows per lane, which share the reads of k and q, from 32 K rows on (128 x 128 at 16
// steps, us, one and two rows: 96 heads 11.3 and 12.9, 256 heads 23.7 and 21.5, 1024 heads 77 and 69; 64 x 64, 512 heads 12.9 and 13.2,
// 1024 heads 22.3 and 21.2).
template <bool BLOCK>
const void* forward_rows_for(int state_dtype, int slots, int Hv, int Dk, int Dv, int* rows) {
  const bool many = (long long)slots * Hv * Dv >= 32768;
  return state_dtype == DFLASH_BF16   ? forward_rows_for<DFLASH_BF16, BLOCK>(Dk, Dv, many, rows)
         : state_dtype == DFLASH_FP16 ? forward_rows_for<DFLASH_FP16, BLOCK>(Dk, Dv, many, rows)
                                      : forward_rows_for<DFLASH_FP32, BLOCK>(Dk, Dv, many, rows);
}

// ---------------------------------------------------------------------------
// Dk = Dv = 128, T <= 16, one gate per head, fp32 state: the block in closed form.
// With c_t = prod_{u<=t} g_u (masked steps: g = 1, beta = 0) the recurrence unrolls to
//     kv_t    = c_t (S0 k_t) + sum_{s<t}  (c_t/c_s) (k_s.k_t) delta_s
//     delta_t = beta_t (v_t - kv_t)
//     y_t     = c_t (S0 q_t) + sum_{s<=t} (c_t/c_s) (k_s.q_t) delta_s
//     S_T     = c_T S0 + sum_s (c_T/c_s) delta_s (x) k_s
// In matrix form, with U = S0 K^T, W = S0 Q^T (Dv x T), L[t][s] = beta_t (c_t/c_s)(k_s.k_t) for
// s < t and Lq[t][s] = (c_t/c_s)(k_s.q_t) for s <= t:
//     Delta = R (I + L)^-T with R[dv][t] = beta_t (v_t[dv] - c_t U[dv][t]),
//     Y = c W + Delta Lq^T,     S_T^T = c_T S0^T + K^T diag(c_T/c_s) Delta^T.
// Every product runs on the matrix cores (v_mfma_f32_16x16x4_f32; with bf16 q and k the three
// big ones on the bf16 matrix cores, see split_bf16); the only serial part
// is the inverse of the T x T unit triangular matrix, once per head.  The arithmetic per
// state element drops from ~5 T vector operations to ~1.5 T matrix-core operations, which
// leaves the kernel bound by the state traffic.
//
// MFMA 16x16x4 lanes: A lane l holds A[i = l % 16][k = l / 16], B lane l holds B[k = l / 16]
// [j = l % 16], accumulator register r of lane l is C[4 (l / 16) + r][l % 16].
// Lane (li = lane % 16, kq = lane / 16) of wave w keeps S rows 32w + 16a + li (a = 0, 1),
// columns 16c + 4kq + e (c = 0..7, e = 0..3).  As the A operand of S0 K^T, component e of
// chunk c pairs with k_t[16c + 4kq + e] on the B side: the columns are only summed in another
// order.  As the accumulator of the transposed update (rows = Dk, columns = Dv) the same
// registers are C[16c + 4kq + e][row li], so the new state lands where the old one was.
// ---------------------------------------------------------------------------
constexpr int kKPad = 132;  // row pitch of K and Q in LDS, in floats
constexpr int kRPad = 17;   // row pitch of R
constexpr int kOffK = 0;
constexpr int kOffQ = kOffK + 16 * kKPad;  // Q, then Delta[t][dv]
constexpr int kOffV = kOffQ + 16 * kKPad;
constexpr int kOffR = kOffV + 16 * 128;
constexpr int kOffRat = kOffR + 128 * kRPad;  // c_t / c_s, 0 above the diagonal
constexpr int kOffLq = kOffRat + 256;
constexpr int kOffM = kOffLq + 256;  // (I + L)^-1
constexpr int kOffC = kOffM + 256;
constexpr int kOffBeta = kOffC + 16;   // 0 for masked and missing steps
constexpr int kOffGate = kOffBeta + 16;  // 1 for masked and missing steps
constexpr int kOffOn = kOffGate + 16;    // 1 for steps that count, 0 for masked and missing ones
constexpr int kOffSS = kOffOn + 16;      // [tile of 16 rows][step]: its share of a step's sum of squares
constexpr int kChunkLdsFloats = kOffSS + 128;
// Where q, k and v come from: arrays, or the block's projections (gdn_block_device.h).  kThirteenWaves: twelve waves with four steps of q, k or v each, the
// first eight of them with a tile of 16 rows of S as well, and one for what a head has once.  kFourWaves: the four waves of the array form.
enum Source { kFromArrays = 0, kFourWaves, kThirteenWaves };
constexpr int kBlockConvWaves = 12, kBlockThreads = 64 * (kBlockConvWaves + 1), kBlockSteps = 2;
template <Source FROM>
struct BlockIncoming : ConvRows<4, kBlockSteps> {};
template <>
struct BlockIncoming<kFourWaves> {
  ConvRows<8> rows[3];  // q, k, v
  GateBits gates;
};

// Four consecutive elements at element i (a multiple of 4) of a 16-byte aligned array.
__device__ __forceinline__ void store4_from_f32(void* p, size_t i, f32x4_t v, int dt) {
  if (dt == DFLASH_FP32) {
    *reinterpret_cast<f32x4_t*>((float*)p + i) = v;
  } else if (dt == DFLASH_BF16) {
    *reinterpret_cast<uint2*>((uint16_t*)p + i) = uint2{f32_to_bf16_bits(v.x) | (f32_to_bf16_bits(v.y) << 16),
                                                        f32_to_bf16_bits(v.z) | (f32_to_bf16_bits(v.w) << 16)};
  } else {
    *reinterpret_cast<uint2*>((uint16_t*)p + i) = uint2{f32_to_f16_bits(v.x) | (f32_to_f16_bits(v.y) << 16),
                                                        f32_to_f16_bits(v.z) | (f32_to_f16_bits(v.w) << 16)};
  }
}
// The same for values that already are representable in dt (the bits are taken, not rounded).
__device__ __forceinline__ void store4_rounded(void* p, size_t i, f32x4_t v, int dt) {
  if (dt == DFLASH_BF16) {
    *reinterpret_cast<uint2*>((uint16_t*)p + i) =
        uint2{(__float_as_uint(v.x) >> 16) | (__float_as_uint(v.y) & 0xffff0000u),
              (__float_as_uint(v.z) >> 16) | (__float_as_uint(v.w) & 0xffff0000u)};
  } else {
    store4_from_f32(p, i, v, dt);
  }
}
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
__device__ __forceinline__ f32x4_t mfma32_bf16(const uint32_t (&a)[4], const uint32_t (&b)[4], f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, uint4{a[0], a[1], a[2], a[3]}),
                                                 __builtin_bit_cast(bf16x8_t, uint4{b[0], b[1], b[2], b[3]}), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma16_bf16(const uint32_t (&a)[2], const uint32_t (&b)[2], f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_t, uint2{a[0], a[1]}),
                                                   __builtin_bit_cast(s16x4_t, uint2{b[0], b[1]}), c, 0, 0, 0);
}

// What one (slot, head) item brings in from memory, as it sits in registers while in flight.
template <bool WIDE, int TILES>
struct Incoming {
  Raw8<WIDE> k, q, v;
  uint32_t gate_bits, beta_bits, mask_byte;  // of step tid (threads below 16), as loaded
  // fused output norm: this lane's four columns of z (step li) and of the norm weight per row tile
  uint2 z2[TILES], w2[TILES];    // 16-bit elements
  f32x4_t z4[TILES], w4[TILES];  // fp32 elements
  f32x4_t st[TILES][8];
};
// Channel `at` of the head in q (0), k (1) or v (2).
__device__ __forceinline__ int block_channel(const GdnArgs& a, int which, int hv, int hk, int at) {
  return (which == 0 ? hk : which == 1 ? a.Hk + hk : 2 * a.Hk + hv) * 128 + at;
}
// First step of a lane of the wide form
__device__ __forceinline__ int block_step(int wave, int lane) { return 4 * (wave & 3) + kBlockSteps * (lane >> 5); }
template <bool WIDE, bool NORM, Source FROM, int TILES>
__device__ __forceinline__ void issue_item_loads(const GdnArgs& a, int item, int tid, Incoming<WIDE, TILES>& in, BlockIncoming<FROM>& block) {
  const int T = a.T;
  const int slot = a.heads.quotient(item), hv = item - slot * a.Hv, hk = a.group.quotient(hv);
  const size_t slotT = (size_t)slot * T;
  const int lane = tid & 63, wave = FROM != kFromArrays ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6, li = lane & 15, kq = lane >> 4;
  // the block's operands first, the state behind them: loads complete in order
#pragma unroll
  for (int j = 0; j < (WIDE ? 2 : 1); ++j) in.k.w[j] = in.q.w[j] = in.v.w[j] = uint4{0u, 0u, 0u, 0u};
  const int t = tid >> 4, seg = tid & 15;
  if constexpr (FROM == kThirteenWaves) {
    request_rows(a.block, slot, block_step(wave, lane), T, (2 * a.Hk + a.Hv) * 128, block_channel(a, wave >> 2, hv, hk, 4 * (lane & 31)), block);
    if (wave >= 8) return;  // (no rows of S)
  } else if constexpr (FROM == kFourWaves) {
#pragma unroll
    for (int j = 0; j < 3; ++j)
      request_rows(a.block, slot, T <= 4 ? lane >> 4 : t, T, (2 * a.Hk + a.Hv) * 128, block_channel(a, j, hv, hk, 8 * seg), block.rows[j]);
    block.gates = request_gates(a.block, slot, lane < T ? lane : T - 1, hv);
  } else if (t < T) {
    const size_t kq_at = ((slotT + t) * a.Hk + hk) * 128 + 8 * seg;
    const size_t v_at = ((slotT + t) * a.Hv + hv) * 128 + 8 * seg;
    in.k = load8_raw<WIDE>(a.k, kq_at);
    in.q = load8_raw<WIDE>(a.q, kq_at);
    in.v = load8_raw<WIDE>(a.v, v_at);
  }
  // gate, beta and mask of step tid as raw bits: whether the step counts is decided once the
  // state has been asked for, so that no request waits for another one's answer
  in.gate_bits = in.beta_bits = 0u;
  in.mask_byte = 1u;
  if (FROM == kFromArrays && tid < T && tid < 16) {
    const size_t at = (slotT + tid) * a.Hv + hv;
    if (a.g_dtype == DFLASH_FP32) {
      in.gate_bits = ((const uint32_t*)a.g)[at];
    } else {
      in.gate_bits = ((const uint16_t*)a.g)[at];
    }
    if (a.beta_dtype == DFLASH_FP32) {
      in.beta_bits = ((const uint32_t*)a.beta)[at];
    } else {
      in.beta_bits = ((const uint16_t*)a.beta)[at];
    }
    if (a.mask != nullptr) in.mask_byte = a.mask[slotT + tid];
  }
  if (NORM) {
    // ahead of the state, like every load whose width depends on a dtype: behind it, the branch
    // around such a load would leave the number of loads in flight unknown at the first wait
    const int tz = li < T ? li : T - 1;
    const size_t zb = (size_t)slot * a.z_batch + (size_t)tz * a.z_row + (size_t)hv * 128;
    const bool wwide = a.weight_dtype == DFLASH_FP32;
#pragma unroll
    for (int t2 = 0; t2 < TILES; ++t2) {
      const int col = 16 * (TILES * wave + t2) + 4 * kq;
      if (WIDE) {
        in.z4[t2] = *reinterpret_cast<const f32x4_t*>((const float*)a.z + zb + col);
      } else {
        in.z2[t2] = *reinterpret_cast<const uint2*>((const uint16_t*)a.z + zb + col);
      }
      if (wwide) {
        in.w4[t2] = *reinterpret_cast<const f32x4_t*>((const float*)a.norm_weight + col);
      } else {
        in.w2[t2] = *reinterpret_cast<const uint2*>((const uint16_t*)a.norm_weight + col);
      }
    }
  }
  const f32x4_t* src = reinterpret_cast<const f32x4_t*>((const float*)a.state_in + (size_t)item * 128 * 128);
#pragma unroll
  for (int t2 = 0; t2 < TILES; ++t2)
#pragma unroll
    for (int c = 0; c < 8; ++c)
      in.st[t2][c] = __builtin_nontemporal_load(&src[memory_index((TILES * wave + t2) >> 1, li, kq, (TILES * wave + t2) & 1, c)]);
  // Fence: everything above is on its way before the first of these values is looked at.
  asm volatile("" : "+v"(in.gate_bits), "+v"(in.beta_bits), "+v"(in.mask_byte)::"memory");
}
// Element j = 4h + e (h = 0, 1) of a lane's operand is column 16 (2C + h) + 4kq + e: the 32
// columns 32C .. 32C + 31 over the four lane groups, the same on both sides of a product.
__device__ __forceinline__ void block_operands(const float* sK, const float* sQ, int li, int kq, int C, uint32_t (&kb)[4], uint32_t (&qb)[4]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float4 kf4 = *reinterpret_cast<const float4*>(sK + li * kKPad + 16 * (2 * C + h) + 4 * kq);
    const float4 qf4 = *reinterpret_cast<const float4*>(sQ + li * kKPad + 16 * (2 * C + h) + 4 * kq);
    kb[2 * h] = upper_halves(kf4.x, kf4.y), kb[2 * h + 1] = upper_halves(kf4.z, kf4.w);
    qb[2 * h] = upper_halves(qf4.x, qf4.y), qb[2 * h + 1] = upper_halves(qf4.z, qf4.w);
  }
}
// A barrier that does not wait for memory: __syncthreads() would, for the state on its way in and every store on its way out.
__device__ __forceinline__ void bare_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory"); }
// c_t / c_s = prod_{s < u <= t} g_u for s <= t at 16 t + s, and c_t itself
__device__ __forceinline__ void gate_ratios(const float* sGate, float* sRat, float* sC, int at) {
  const int t = at >> 4, sx = at & 15;
  float gates[16];
#pragma unroll
  for (int u = 0; u < 16; u += 4) {
    const float4 g4 = *reinterpret_cast<const float4*>(sGate + u);
    gates[u] = g4.x, gates[u + 1] = g4.y, gates[u + 2] = g4.z, gates[u + 3] = g4.w;
  }
  float r = sx <= t ? 1.f : 0.f;
#pragma unroll
  for (int u = 1; u < 16; ++u) r *= (u > sx && u <= t) ? gates[u] : 1.f;
  sRat[at] = r;
  if (sx == 0) sC[t] = r * gates[0];
}
// M = (I + L)^-1 by forward substitution, column li per lane.  L[t][s] sits in lane 16 (s / 4) + t, register s % 4 of this wave and
// reaches the others through v_readlane.
__device__ __forceinline__ void unit_inverse(const float (&Lr)[4], float* sM, int li, int kq) {
  float x[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) x[t] = t == li ? 1.f : 0.f;
#pragma unroll
  for (int sx = 0; sx < 16; ++sx) {
    if (kq == 0) sM[sx * 16 + li] = x[sx];
#pragma unroll
    for (int t = sx + 1; t < 16; ++t)
      x[t] -= __int_as_float(__builtin_amdgcn_readlane(__float_as_int(Lr[sx & 3]), 16 * (sx >> 2) + t)) * x[sx];
  }
}
// kThirteenWaves: the wave without rows of S.  Gates, beta and their ratios while the others have the conv, Lq and M while they have the products
// with S0; two barriers, which the others meet it at.
__device__ __forceinline__ void block_gates(const GdnArgs& a, int slot, int hv, int lane, float* smem) {
  const int T = a.T, li = lane & 15, kq = lane >> 4;
  float* const sK = smem + kOffK;
  float* const sQ = smem + kOffQ;
  float* const sRat = smem + kOffRat;
  float* const sGate = smem + kOffGate;
  __builtin_amdgcn_s_setprio(3);  // the longest chain of the head
  const GateBits bits = request_gates(a.block, slot, lane < T ? lane : T - 1, hv);
  if (lane < 16) {
    const float g = lane < T ? gate_of(a.block, bits) : 1.f;
    if (lane < T && a.block.g_out != nullptr) a.block.g_out[((size_t)slot * T + lane) * a.Hv + hv] = g;
    sGate[lane] = g;
    smem[kOffBeta + lane] = lane < T ? beta_of(bits) : 0.f;
    smem[kOffOn + lane] = lane < T ? 1.f : 0.f;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) gate_ratios(sGate, sRat, smem + kOffC, 64 * i + lane);
  bare_barrier();
  f32x4_t kk = {0.f, 0.f, 0.f, 0.f}, kq_sum = {0.f, 0.f, 0.f, 0.f};  // [s][t] = k_s . k_t and k_s . q_t
#pragma unroll
  for (int C = 0; C < 4; ++C) {
    uint32_t kb[4], qb[4];
    block_operands(sK, sQ, li, kq, C, kb, qb);
    kk = mfma32_bf16(kb, kb, kk);
    kq_sum = mfma32_bf16(kb, qb, kq_sum);
  }
  const float bt = smem[kOffBeta + li];
  float Lr[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int sx = 4 * kq + r;
    const float rat = sRat[li * 16 + sx];  // 0 for s > t
    Lr[r] = sx < li ? bt * rat * kk[r] : 0.f;
    smem[kOffLq + li * 16 + sx] = rat * kq_sum[r];
  }
  unit_inverse(Lr, smem + kOffM, li, kq);
  bare_barrier();
}
// One workgroup per (slot, head); the register cap keeps at least three on a compute unit, two (kFourWaves) or one (kThirteenWaves).
// SPLIT: q and k are bf16 arrays; the products with S0 and the state update run on the bf16
// matrix cores with the fp32 factor in three exact pieces (see split_bf16).
// kFourWaves, kThirteenWaves: q, k, v, the gates and beta are made here, from the block's projections (gdn_block_device.h), while the state is on its
// way.  A launch of the prepare kernel before this one took 5.4 us for what is 0.4 MB, and a microsecond to the next.  In an ordinary block 32 of
// 256 compute units have a head to work on and nothing beside it, so what counts is the longest chain of a head: eight waves with a tile of rows each, two to a
// SIMD, fill each other's waits, four more share the conv with them, and one has what a head has once, gates, ratios and (I + L)^-1, beside the
// conv and the products with S0.  16 tokens of 32 heads 16.9 (four waves of two tiles, the second of them with the inverse) -> 13.8 -> 13.1 us
// (a wave loads the rows and taps of one of q, k, v instead of all three) -> 12.6 (sums over lanes without LDS, two roundings to a conversion, the roots
// of two steps at once: three waves of a SIMD share the issue port for the 2.3 us of the conv, 400 vector instructions each).  The state asked for
// behind everybody's conv operands instead of behind one's own: 12.8.  Thirteen waves leave no room for a second head on the compute unit;
// where there are more heads than compute units the four waves of kFourWaves, two heads at a time, are faster (dflash_gdn_block says from where on).
template <bool WIDE, bool NORM, bool SPLIT, Source FROM>
__global__ __launch_bounds__(FROM == kThirteenWaves ? kBlockThreads : kThreads)
__attribute__((amdgpu_waves_per_eu(FROM == kThirteenWaves ? 4 : FROM == kFourWaves ? 2 : 3, FROM == kThirteenWaves ? 4 : FROM == kFourWaves ? 2 : 3)))
void gdn_forward_chunk_128(GdnArgs a) {
  const int in_dtype = FROM != kFromArrays || SPLIT ? DFLASH_BF16 : a.in_dtype;
  constexpr int TILES = FROM == kThirteenWaves ? 1 : 2;  // of 16 rows of S to a wave
  extern __shared__ __align__(16) float smem[];
  float* sK = smem + kOffK;
  float* sQ = smem + kOffQ;
  float* sD = smem + kOffQ;
  float* sV = smem + kOffV;
  float* sR = smem + kOffR;
  float* sRat = smem + kOffRat;
  float* sLq = smem + kOffLq;
  float* sM = smem + kOffM;
  float* sC = smem + kOffC;
  float* sBeta = smem + kOffBeta;
  float* sGate = smem + kOffGate;
  float* sOn = smem + kOffOn;
  float* sSS = smem + kOffSS;

  const int T = a.T;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: branches on it are real branches
  const int li = lane & 15, kq = lane >> 4;

  const int item = blockIdx.x;
  const int slot = a.heads.quotient(item), hv = item - slot * a.Hv;
  const size_t slotT = (size_t)slot * T;
  if constexpr (FROM == kThirteenWaves) {
    if (wave == kBlockConvWaves) {
      block_gates(a, slot, hv, lane, smem);
      return;
    }
  }
  Incoming<WIDE, TILES> cur;
  BlockIncoming<FROM> block;
  issue_item_loads<WIDE, NORM, FROM, TILES>(a, item, tid, cur, block);
  const size_t sbase = (size_t)item * 128 * 128;
  f32x4_t (&st)[TILES][8] = cur.st;
  uint2 (&z2)[TILES] = cur.z2, (&w2)[TILES] = cur.w2;
  f32x4_t (&z4)[TILES] = cur.z4, (&w4)[TILES] = cur.w4;
  if constexpr (FROM == kThirteenWaves) {
    const int seg = lane & 31, hk = a.group.quotient(hv), C = (2 * a.Hk + a.Hv) * 128;
    const int which = wave >> 2, t = block_step(wave, lane);
    float* const dst = which == 0 ? sQ : which == 1 ? sK : sV;
    const int pitch = which == 2 ? 128 : kKPad;
    float x[kBlockSteps][4] = {};
    if (4 * (wave & 3) < T) {
      const bool keeps = which == 2 || hv == hk * (int)a.group.by;  // a key head's: by the first of its value heads
      convolve(a.block, slot, t, T, C, block_channel(a, which, hv, hk, 4 * seg), keeps, block, x);
      if (which < 2) {
        const float scale = which == 1 ? a.block.scale_k : a.block.scale_q;
        static_assert(kBlockSteps == 2, "two rows at a time");
        normalise<4, 32>(x, scale, a.block.eps);
      }
      if (which == 1 && keeps && a.block.k_out != nullptr) {
#pragma unroll
        for (int i = 0; i < kBlockSteps; ++i)
          if (t + i < T) store_exact<4>(a.block.k_out + ((slotT + t + i) * a.Hk + hk) * 128 + 4 * seg, x[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kBlockSteps; ++i)
      *reinterpret_cast<f32x4_t*>(dst + (t + i) * pitch + 4 * seg) =
          t + i < T ? f32x4_t{x[i][0], x[i][1], x[i][2], x[i][3]} : f32x4_t{0.f, 0.f, 0.f, 0.f};
  } else if constexpr (FROM == kFourWaves) {
    const int seg = tid & 15, hk = a.group.quotient(hv), C = (2 * a.Hk + a.Hv) * 128;
    // every wave its four steps of q, k and v, of up to four steps in all one of the three
    const bool few = T <= 4;
    const int t = few ? lane >> 4 : tid >> 4;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      float* const dst = j == 0 ? sQ : j == 1 ? sK : sV;
      const int pitch = j == 2 ? 128 : kKPad;
      float all[1][8] = {};
      auto& x = all[0];
      if (few ? wave == j : 4 * wave < T) {
        const bool keeps = j == 2 || hv == hk * (int)a.group.by;  // a key head's: by the first of its value heads
        convolve(a.block, slot, t, T, C, block_channel(a, j, hv, hk, 8 * seg), keeps, block.rows[j], all);
        if (j < 2) normalise<8, 16>(x, j == 1 ? a.block.scale_k : a.block.scale_q, a.block.eps);
        if (j == 1 && keeps && t < T && a.block.k_out != nullptr)
          store_exact<8>(a.block.k_out + ((slotT + t) * a.Hk + hk) * 128 + 8 * seg, x);
      }
      const auto put = [&](int step, bool on) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; e += 4)
          *reinterpret_cast<f32x4_t*>(dst + step * pitch + 8 * seg + e) =
              on ? f32x4_t{x[e], x[e + 1], x[e + 2], x[e + 3]} : f32x4_t{0.f, 0.f, 0.f, 0.f};
      };
      if (!few) {
        put(t, t < T);
      } else if (wave == j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) put(4 * i + t, i == 0 && t < T);
      }
    }
    if (wave == 3 && lane < 16) {
      const float g = lane < T ? gate_of(a.block, block.gates) : 1.f;
      if (lane < T && a.block.g_out != nullptr) a.block.g_out[(slotT + lane) * a.Hv + hv] = g;
      sGate[lane] = g;
      sBeta[lane] = lane < T ? beta_of(block.gates) : 0.f;
      sOn[lane] = lane < T ? 1.f : 0.f;
    }
  } else {
    const int t = tid >> 4, seg = tid & 15;
    raw8_to_lds(cur.k, in_dtype, sK + t * kKPad + 8 * seg);
    raw8_to_lds(cur.q, in_dtype, sQ + t * kKPad + 8 * seg);
    raw8_to_lds(cur.v, in_dtype, sV + t * 128 + 8 * seg);
  }
  if (FROM == kFromArrays && tid < 16) {
    const bool on = tid < T && cur.mask_byte != 0;  // masked and missing steps: gate 1, beta 0
    sGate[tid] = on ? bits_as_f32(cur.gate_bits, a.g_dtype) : 1.f;
    sBeta[tid] = on ? bits_as_f32(cur.beta_bits, a.beta_dtype) : 0.f;
    sOn[tid] = on ? 1.f : 0.f;
  }
  if constexpr (FROM == kThirteenWaves) {
    bare_barrier();  // (nobody waits for the state here)
    if (wave >= 8) return;
  } else {
    __syncthreads();
    gate_ratios(sGate, sRat, sC, tid);
    __syncthreads();
  }

  // ---- U = S0 K^T, W = S0 Q^T (every wave, its 32 rows); K K^T (wave 1), K Q^T (wave 2) -------
#pragma unroll
  for (int t2 = 0; t2 < TILES; ++t2)
#pragma unroll
    for (int m = 0; m < 4; ++m) swap_row_bit(st[t2][2 * m], st[t2][2 * m + 1]);
  f32x4_t U[TILES], W[TILES], X = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t2 = 0; t2 < TILES; ++t2) U[t2] = f32x4_t{0.f, 0.f, 0.f, 0.f}, W[t2] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if constexpr (SPLIT) {
#pragma unroll
    for (int C = 0; C < 4; ++C) {
      uint32_t kb[4], qb[4];
      block_operands(sK, sQ, li, kq, C, kb, qb);
#pragma unroll
      for (int t2 = 0; t2 < TILES; ++t2) {
        const float f[8] = {st[t2][2 * C][0],     st[t2][2 * C][1],     st[t2][2 * C][2],     st[t2][2 * C][3],
                            st[t2][2 * C + 1][0], st[t2][2 * C + 1][1], st[t2][2 * C + 1][2], st[t2][2 * C + 1][3]};
        const Pieces<8> sp = split_bf16(f);
        U[t2] = mfma32_bf16(sp.lo, kb, U[t2]);
        W[t2] = mfma32_bf16(sp.lo, qb, W[t2]);
        U[t2] = mfma32_bf16(sp.mid, kb, U[t2]);
        W[t2] = mfma32_bf16(sp.mid, qb, W[t2]);
        U[t2] = mfma32_bf16(sp.hi, kb, U[t2]);
        W[t2] = mfma32_bf16(sp.hi, qb, W[t2]);
      }
      if (FROM != kThirteenWaves && wave == 1) X = mfma32_bf16(kb, kb, X);  // [s][t] = k_s . k_t
      if (FROM != kThirteenWaves && wave == 2) X = mfma32_bf16(kb, qb, X);  // [s][t] = k_s . q_t
    }
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float4 kf4 = *reinterpret_cast<const float4*>(sK + li * kKPad + 16 * c + 4 * kq);
      const float4 qf4 = *reinterpret_cast<const float4*>(sQ + li * kKPad + 16 * c + 4 * kq);
      const float kf[4] = {kf4.x, kf4.y, kf4.z, kf4.w};
      const float qf[4] = {qf4.x, qf4.y, qf4.z, qf4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int t2 = 0; t2 < TILES; ++t2) {
          U[t2] = mfma4(st[t2][c][e], kf[e], U[t2]);
          W[t2] = mfma4(st[t2][c][e], qf[e], W[t2]);
        }
        if (wave == 1) X = mfma4(kf[e], kf[e], X);  // [s][t] = k_s . k_t
        if (wave == 2) X = mfma4(kf[e], qf[e], X);  // [s][t] = k_s . q_t
      }
    }
  }
  {
    const int t = li;
    const float ct = sC[t], bt = sBeta[t];
    float Lr[4];  // wave 1: L[t][4kq + r], wave 2: Lq[t][4kq + r]
    if constexpr (FROM != kThirteenWaves) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int sx = 4 * kq + r;
        const float rat = sRat[t * 16 + sx];  // 0 for s > t
        Lr[r] = wave == 1 ? (sx < t ? bt * rat * X[r] : 0.f) : rat * X[r];
        if (wave == 2) sLq[t * 16 + sx] = Lr[r];
      }
    }
#pragma unroll
    for (int t2 = 0; t2 < TILES; ++t2) {
      const int row0 = 16 * (TILES * wave + t2) + 4 * kq;
      const float4 v4 = *reinterpret_cast<const float4*>(sV + t * 128 + row0);
      sR[(row0 + 0) * kRPad + t] = bt * (v4.x - ct * U[t2][0]);
      sR[(row0 + 1) * kRPad + t] = bt * (v4.y - ct * U[t2][1]);
      sR[(row0 + 2) * kRPad + t] = bt * (v4.z - ct * U[t2][2]);
      sR[(row0 + 3) * kRPad + t] = bt * (v4.w - ct * U[t2][3]);
    }
    if (FROM != kThirteenWaves && wave == 1) unit_inverse(Lr, sM, li, kq);
  }
  if constexpr (FROM == kThirteenWaves) bare_barrier();
  else __syncthreads();
  // Lq, R and M are complete; nobody reads Q any more

  // ---- Delta = R M^T: rows of this wave, accumulator (row 4kq + r, column t = li) ---------------
  f32x4_t D[TILES];
#pragma unroll
  for (int t2 = 0; t2 < TILES; ++t2) {
    D[t2] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      D[t2] = mfma4(sR[(16 * (TILES * wave + t2) + li) * kRPad + 4 * j + kq], sM[li * 16 + 4 * j + kq], D[t2]);
  }
  const size_t obase = ((slotT + li) * a.Hv + hv) * 128;  // step li of this head in y and the tape
#pragma unroll
  for (int t2 = 0; t2 < TILES; ++t2) {
    const int row0 = 16 * (TILES * wave + t2) + 4 * kq;
    *reinterpret_cast<f32x4_t*>(sD + li * 128 + row0) = D[t2];
  }
  if constexpr (FROM == kThirteenWaves) {
    if (li < T) *reinterpret_cast<f32x4_t*>(a.tape + obase + 16 * wave + 4 * kq) = D[0];
  } else {
    // the tape leaves from LDS in full 128-byte lines: lane (t, q) stores this wave's rows
    // 32 wave + 8 q ..+7 of step t (the matrix-core layout would give 64-byte pieces)
    const int t = lane >> 2, dv0 = 32 * wave + 8 * (lane & 3);
    if (t < T) {
      float* dst = a.tape + ((slotT + t) * a.Hv + hv) * 128 + dv0;
      *reinterpret_cast<f32x4_t*>(dst) = *reinterpret_cast<const f32x4_t*>(sD + t * 128 + dv0);
      *reinterpret_cast<f32x4_t*>(dst + 4) = *reinterpret_cast<const f32x4_t*>(sD + t * 128 + dv0 + 4);
    }
  }
  // (a wave reads the rows of Delta that it has written)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  // ---- Y = c W + Delta Lq^T -----------------------------------------------------------------------
  float Yn[TILES][4];  // fused norm: Y rounded to the array dtype, kept until every wave's sum of squares is in
  float dA[TILES][4];  // Delta[row 16 t2 + li][s = 4j + kq]
#pragma unroll
  for (int t2 = 0; t2 < TILES; ++t2)
#pragma unroll
    for (int j = 0; j < 4; ++j) dA[t2][j] = sD[(4 * j + kq) * 128 + 16 * (TILES * wave + t2) + li];
  {
    const float ct = sC[li];
    const bool on = sOn[li] != 0.f;
#pragma unroll
    for (int t2 = 0; t2 < TILES; ++t2) {
      f32x4_t Y = W[t2] * ct;
#pragma unroll
      for (int j = 0; j < 4; ++j) Y = mfma4(dA[t2][j], sLq[li * 16 + 4 * j + kq], Y);
      if (!on) Y = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (!NORM) {
        if (li < T) store4_from_f32(a.y, obase + 16 * (TILES * wave + t2) + 4 * kq, Y, in_dtype);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) Yn[t2][r] = round_through(Y[r], in_dtype);  // the recurrence's output, as an array
      }
    }
    if (NORM) {
      // a tile's 16 columns of step li: 4 per lane, the four lanes (li, kq) of a step added up
#pragma unroll
      for (int t2 = 0; t2 < TILES; ++t2) {
        float ss = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) ss += Yn[t2][r] * Yn[t2][r];
        ss = plus_far(ss, true);
        if (kq == 0) sSS[16 * (TILES * wave + t2) + li] = ss;  // read after the state update, behind its barrier
      }
    }
  }

  // ---- S_T^T = c_T S0^T + K^T diag(c_T / c_s) Delta^T -----------------------------------------------
  {
    const float cT = sC[T - 1];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float cf = sRat[(T - 1) * 16 + 4 * j + kq];  // 0 beyond step T - 1
#pragma unroll
      for (int t2 = 0; t2 < TILES; ++t2) dA[t2][j] *= cf;
    }
    Pieces<4> dp[TILES];  // SPLIT: the scaled Delta in pieces; element j of a lane's operand is step 4j + kq
    if constexpr (SPLIT) {
#pragma unroll
      for (int t2 = 0; t2 < TILES; ++t2) dp[t2] = split_bf16(dA[t2]);
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      float kA[4];  // K[s = 4j + kq][16c + li]
#pragma unroll
      for (int j = 0; j < 4; ++j) kA[j] = sK[(4 * j + kq) * kKPad + 16 * c + li];
      const uint32_t ka[2] = {upper_halves(kA[0], kA[1]), upper_halves(kA[2], kA[3])};
#pragma unroll
      for (int t2 = 0; t2 < TILES; ++t2) {
        f32x4_t acc = st[t2][c] * cT;
        if constexpr (SPLIT) {
          acc = mfma16_bf16(ka, dp[t2].lo, acc);
          acc = mfma16_bf16(ka, dp[t2].mid, acc);
          acc = mfma16_bf16(ka, dp[t2].hi, acc);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) acc = mfma4(kA[j], dA[t2][j], acc);
        }
        st[t2][c] = acc;
      }
    }
  }
  if (NORM) {
    // silu(z) * rms_norm(y, weight) with the rounding points of the separate operators: y, the
    // normalised and weighted y, sigmoid(z), z * sigmoid(z) and the product are arrays of the
    // input dtype; sums and the reciprocal root are fp32.
    // a bare barrier: __syncthreads() would also wait until every store issued so far has been
    // acknowledged, and the stores of the state are about to follow
    bare_barrier();
    float total = sSS[li];
#pragma unroll
    for (int i = 1; i < 8; ++i) total += sSS[16 * i + li];
    float zf[TILES][4], wf[TILES][4];
#pragma unroll
    for (int t2 = 0; t2 < TILES; ++t2) {
      if (WIDE) {
#pragma unroll
        for (int r = 0; r < 4; ++r) zf[t2][r] = z4[t2][r];
      } else {
        const uint32_t h[4] = {z2[t2].x & 0xFFFFu, z2[t2].x >> 16, z2[t2].y & 0xFFFFu, z2[t2].y >> 16};
#pragma unroll
        for (int r = 0; r < 4; ++r) zf[t2][r] = bits_as_f32(h[r], in_dtype);
      }
      if (a.weight_dtype == DFLASH_FP32) {
#pragma unroll
        for (int r = 0; r < 4; ++r) wf[t2][r] = w4[t2][r];
      } else {
        const uint32_t h[4] = {w2[t2].x & 0xFFFFu, w2[t2].x >> 16, w2[t2].y & 0xFFFFu, w2[t2].y >> 16};
#pragma unroll
        for (int r = 0; r < 4; ++r) wf[t2][r] = bits_as_f32(h[r], a.weight_dtype);
      }
    }
    // A head's launch occupies one compute unit in eight, so whatever this tail costs per lane is
    // added to the layer's latency in full: the 16-bit dtypes take the hardware's exp2,
    // reciprocal and reciprocal root (each within an ulp of fp32, far below half an ulp of a
    // 16-bit array) and a rounding written out for the dtype; fp32 arrays keep the library forms.
    auto finish = [&](auto rnd, auto sigmoid, float inv_rms) __attribute__((always_inline)) {
#pragma unroll
      for (int t2 = 0; t2 < TILES; ++t2) {
        f32x4_t o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float normed = rnd(Yn[t2][r] * inv_rms * wf[t2][r]);
          o[r] = rnd(rnd(zf[t2][r] * rnd(sigmoid(zf[t2][r]))) * normed);
        }
        if (li < T) store4_rounded(a.y, obase + 16 * (TILES * wave + t2) + 4 * kq, o, in_dtype);
      }
    };
    auto fast_sigmoid = [](float x) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * x)); };
    if (in_dtype == DFLASH_BF16) {
      finish([](float v) { uint32_t u = __float_as_uint(v); u += 0x7fffu + ((u >> 16) & 1u); return __uint_as_float(u & 0xffff0000u); },
             fast_sigmoid, __builtin_amdgcn_rsqf(total * (1.0f / 128.0f) + a.eps));
    } else if (in_dtype == DFLASH_FP16) {
      finish([](float v) { return (float)(_Float16)v; }, fast_sigmoid, __builtin_amdgcn_rsqf(total * (1.0f / 128.0f) + a.eps));
    } else {
      finish([](float v) { return v; }, [](float x) { return 1.0f / (1.0f + expf(-x)); },
             1.0f / sqrtf(total / 128.0f + a.eps));
    }
  }
  {
    f32x4_t* out = reinterpret_cast<f32x4_t*>((float*)a.state_out + sbase);
#pragma unroll
    for (int t2 = 0; t2 < TILES; ++t2)
#pragma unroll
      for (int m = 0; m < 4; ++m) swap_row_bit(st[t2][2 * m], st[t2][2 * m + 1]);
#pragma unroll
    for (int t2 = 0; t2 < TILES; ++t2)
#pragma unroll
      for (int c = 0; c < 8; ++c)
        __builtin_nontemporal_store(st[t2][c], &out[memory_index((TILES * wave + t2) >> 1, li, kq, (TILES * wave + t2) & 1, c)]);
  }
}

// ---------------------------------------------------------------------------
// Any Dk, Dv: one workgroup per (slot, head), a thread walks whole rows of S, which lives in
// state_out between steps (so it is rounded through the state dtype after every step by
// construction).  Slow and simple; the kernels above have the head sizes of the models served.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void gdn_forward_generic(GdnArgs a) {
  const int slot = blockIdx.x / a.Hv, hv = blockIdx.x % a.Hv;
  const int hk = hv / (a.Hv / a.Hk);
  const size_t slotT = (size_t)slot * a.T;
  const size_t sbase = (size_t)blockIdx.x * a.Dv * a.Dk;
  for (int dv = threadIdx.x; dv < a.Dv; dv += kThreads) {
    const size_t row = sbase + (size_t)dv * a.Dk;
    for (int dk = 0; dk < a.Dk; ++dk)
      store_from_f32(a.state_out, row + dk, load_as_f32(a.state_in, row + dk, a.state_dtype), a.state_dtype);
    for (int t = 0; t < a.T; ++t) {
      const size_t o = ((slotT + t) * a.Hv + hv) * a.Dv + dv;
      float delta = 0.f, y = 0.f;
      if (a.mask == nullptr || a.mask[slotT + t] != 0) {
        const size_t kq0 = ((slotT + t) * a.Hk + hk) * a.Dk;
        const size_t g0 = a.g_per_dk ? ((slotT + t) * a.Hv + hv) * a.Dk : (slotT + t) * a.Hv + hv;
        float kv = 0.f;
        for (int dk = 0; dk < a.Dk; ++dk) {
          const float g = load_as_f32(a.g, a.g_per_dk ? g0 + dk : g0, a.g_dtype);
          kv += load_as_f32(a.state_out, row + dk, a.state_dtype) * g * load_as_f32(a.k, kq0 + dk, a.in_dtype);
        }
        delta = (load_as_f32(a.v, o, a.in_dtype) - kv) * load_as_f32(a.beta, (slotT + t) * a.Hv + hv, a.beta_dtype);
        for (int dk = 0; dk < a.Dk; ++dk) {
          const float g = load_as_f32(a.g, a.g_per_dk ? g0 + dk : g0, a.g_dtype);
          const float s = load_as_f32(a.state_out, row + dk, a.state_dtype) * g +
                          load_as_f32(a.k, kq0 + dk, a.in_dtype) * delta;
          y += s * load_as_f32(a.q, kq0 + dk, a.in_dtype);
          store_from_f32(a.state_out, row + dk, s, a.state_dtype);
        }
      }
      a.tape[o] = delta;
      store_from_f32(a.y, o, y, a.in_dtype);
    }
  }
}

}  // namespace
}  // namespace dflash

namespace dflash {
// gdn_prompt.hip
bool gdn_prompt_covers(int slots, int T, int Hk, int Hv, int Dk, int Dv, int in_dtype, int g_per_dk);
size_t gdn_prompt_workspace_bytes(int slots, int T, int Hk, int Hv, int Dk);
int gdn_prompt_launch(const void* q, const void* k, const void* v, const void* g, const void* beta, const void* state_in,
                      void* state_out, void* y, float* tape, const uint8_t* mask, void* workspace, int slots, int T, int Hk,
                      int Hv, int Dk, int Dv, int g_dtype, int beta_dtype, int state_dtype, hipStream_t s);
// gdn_glue.hip
int gdn_gated_norm_launch(const void* x, const void* z, const void* weight, void* y, int B, int T, int H, int D,
                          long long z_batch, long long z_row, int dtype, int weight_dtype, float eps, hipStream_t stream);

namespace {

// Shared body of the entry points; z == nullptr: no output norm; z_row = 0: z laid out like y.
int gdn_forward_launch(const char* who, const void* q, const void* k, const void* v, const void* g, const void* beta,
                       const void* state_in, void* state_out, void* y, float* tape, const uint8_t* mask,
                       const void* z, const void* norm_weight, int weight_dtype, float eps, int slots, int T, int Hk,
                       int Hv, int Dk, int Dv, int in_dtype, int g_dtype, int beta_dtype, int state_dtype,
                       int g_per_dk, void* stream, void* workspace = nullptr, size_t workspace_bytes = 0, long long z_batch = 0,
                       long long z_row = 0) {
  if (z_row == 0) z_row = (long long)Hv * Dv, z_batch = z_row * T;
  const int z_elem = in_dtype == DFLASH_FP32 ? 4 : 2;
  const bool aligned16 = (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)y | (uintptr_t)tape |
                           (uintptr_t)z | (uintptr_t)norm_weight | (uintptr_t)(z ? (z_batch | z_row) * z_elem : 0)) % 16) == 0;
  const bool no_chunk = option(DFLASH_OPT_GDN_STEP_BY_STEP) != 0;  // (tests of one kernel against the other)
  const bool prompt = workspace != nullptr && aligned16 && !no_chunk && gdn_prompt_covers(slots, T, Hk, Hv, Dk, Dv, in_dtype, g_per_dk) &&
                      (((uintptr_t)state_in | (uintptr_t)state_out | (uintptr_t)workspace) % 16) == 0;
  DFLASH_REQUIRE(q && k && v && g && beta && state_out && y && ((state_in && tape) || prompt), DFLASH_ERR_ARG, "%s: null operand", who);
  DFLASH_REQUIRE(state_in != state_out, DFLASH_ERR_ARG, "%s: state_out must not alias state_in", who);
  auto ok = [](int dt) { return dt == DFLASH_BF16 || dt == DFLASH_FP16 || dt == DFLASH_FP32; };
  DFLASH_REQUIRE(ok(in_dtype) && ok(g_dtype) && ok(beta_dtype) && ok(state_dtype) && (!z || ok(weight_dtype)),
                 DFLASH_ERR_ARG, "%s: unknown dtype code", who);
  DFLASH_REQUIRE(slots >= 0 && T >= 0 && Hk > 0 && Hv > 0 && Dk > 0 && Dv > 0, DFLASH_ERR_SHAPE,
                 "%s: non-positive dimension", who);
  DFLASH_REQUIRE(Hv % Hk == 0, DFLASH_ERR_SHAPE, "%s: cannot align K heads %d to V heads %d", who, Hk, Hv);
  DFLASH_REQUIRE((long long)slots * Hv < (1ll << 31), DFLASH_ERR_SHAPE, "%s: too many (slot, head) pairs", who);
  DFLASH_REQUIRE(!z || (norm_weight && Dv % 64 == 0 && Dv <= 256), DFLASH_ERR_SHAPE,
                 "%s: the output norm needs a weight and a row length that is a multiple of 64 up to 256, got %d", who, Dv);
  DFLASH_REQUIRE(!z || (z_batch >= 0 && z_row >= 0 && (long long)slots * T * Hv < (1ll << 31)), DFLASH_ERR_SHAPE,
                 "%s: z needs non-negative strides and fewer than 2^31 rows", who);
  if (slots == 0) return DFLASH_OK;

  GdnArgs a;
  a.q = q; a.k = k; a.v = v; a.g = g; a.beta = beta; a.state_in = state_in; a.state_out = state_out;
  a.y = y; a.tape = tape; a.mask = mask;
  a.T = T; a.Hk = Hk; a.Hv = Hv; a.Dk = Dk; a.Dv = Dv;
  a.heads = Divisor::of(Hv); a.group = Divisor::of(Hv / Hk); a.row_parts = Divisor::of(1);
  a.in_dtype = in_dtype; a.g_dtype = g_dtype; a.beta_dtype = beta_dtype; a.state_dtype = state_dtype;
  a.g_per_dk = g_per_dk ? 1 : 0;
  a.z = z; a.z_batch = z_batch; a.z_row = z_row; a.norm_weight = norm_weight; a.weight_dtype = weight_dtype; a.eps = eps;

  const dim3 grid((unsigned)(slots * Hv)), block(kThreads);
  hipStream_t s = (hipStream_t)stream;
  a.staged = T < 16 ? T : 16;
  const size_t smem = (size_t)a.staged * (3 * 128 + (g_per_dk ? 128 : 1) + 2) * sizeof(float);
  const bool fast = Dk == 128 && Dv == 128 && T >= 1 &&
                    (state_dtype != DFLASH_FP32 ||
                     (((uintptr_t)state_in % 16) == 0 && ((uintptr_t)state_out % 16) == 0));
  const bool chunk = fast && !g_per_dk && state_dtype == DFLASH_FP32 && T <= 16 && aligned16 && !no_chunk;
  const void* by_rows = nullptr;
  int rows = Dv;
  if (!prompt && !chunk && !g_per_dk && T >= 1 && aligned16 && (((uintptr_t)state_in | (uintptr_t)state_out) % 16) == 0 &&
      !(fast && state_dtype == DFLASH_FP32)) {
    by_rows = forward_rows_for<false>(state_dtype, slots, Hv, Dk, Dv, &rows);
    if ((long long)slots * Hv * (Dv / rows) >= (1ll << 31)) by_rows = nullptr;
  }
  bool norm_done = false;
  if (prompt) {
    const size_t need = gdn_prompt_workspace_bytes(slots, T, Hk, Hv, Dk);
    DFLASH_REQUIRE(workspace_bytes >= need, DFLASH_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, need,
                   workspace_bytes);
    const int rc = gdn_prompt_launch(q, k, v, g, beta, state_in, state_out, y, tape, mask, workspace, slots, T, Hk, Hv, Dk, Dv,
                                     g_dtype, beta_dtype, state_dtype, s);
    if (rc != DFLASH_OK) return rc;
  } else if (chunk) {
    const size_t lds = kChunkLdsFloats * sizeof(float);
    const bool wide = in_dtype == DFLASH_FP32;
    const bool split = in_dtype == DFLASH_BF16;  // q and k are bf16 numbers: exact products on the bf16 matrix cores
    if (z) {
      if (wide) hipLaunchKernelGGL((gdn_forward_chunk_128<true, true, false, kFromArrays>), grid, block, lds, s, a);
      else if (split) hipLaunchKernelGGL((gdn_forward_chunk_128<false, true, true, kFromArrays>), grid, block, lds, s, a);
      else hipLaunchKernelGGL((gdn_forward_chunk_128<false, true, false, kFromArrays>), grid, block, lds, s, a);
      norm_done = true;
    } else {
      if (wide) hipLaunchKernelGGL((gdn_forward_chunk_128<true, false, false, kFromArrays>), grid, block, lds, s, a);
      else if (split) hipLaunchKernelGGL((gdn_forward_chunk_128<false, false, true, kFromArrays>), grid, block, lds, s, a);
      else hipLaunchKernelGGL((gdn_forward_chunk_128<false, false, false, kFromArrays>), grid, block, lds, s, a);
    }
  } else if (by_rows != nullptr) {
    a.row_parts = Divisor::of(Dv / rows);
    void* args[] = {&a};
    DFLASH_HIP_OK(hipLaunchKernel(by_rows, dim3((unsigned)(slots * Hv * (Dv / rows))), block, args, 0, s));
  } else if (fast) {
    if (g_per_dk) {
      hipLaunchKernelGGL((gdn_forward_128<true, false>), grid, block, smem, s, a);
    } else if (state_dtype == DFLASH_FP32) {
      hipLaunchKernelGGL((gdn_forward_128<false, true>), grid, block, smem, s, a);
    } else {
      hipLaunchKernelGGL((gdn_forward_128<false, false>), grid, block, smem, s, a);
    }
  } else {
    hipLaunchKernelGGL(gdn_forward_generic, grid, block, 0, s, a);
  }
  DFLASH_HIP_OK(hipGetLastError());
  if (z && !norm_done)  // the other kernels leave the recurrence's output in y: normalise it in place
    return T == 0 ? DFLASH_OK : gdn_gated_norm_launch(y, z, norm_weight, y, slots, T, Hv, Dv, z_batch, z_row, in_dtype, weight_dtype,
                                                      eps, s);
  return DFLASH_OK;
}

// The value a Python float takes when it meets a bf16 array.
float as_bf16_scalar(double v) {
  const float f = (float)v;
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  u += 0x7fffu + ((u >> 16) & 1u);
  u &= 0xffff0000u;
  float r;
  __builtin_memcpy(&r, &u, 4);
  return r;
}

}  // namespace
}  // namespace dflash

extern "C" int dflash_gdn_block(const dflash_gdn_block_args* p, void* stream) {
  using namespace dflash;
  const char* who = "dflash_gdn_block";
  DFLASH_REQUIRE(p && p->qkv && p->conv_w && p->a && p->b && p->A_log && p->dt_bias && p->conv_next && p->state_in && p->state_out &&
                     p->y && p->tape && (!p->z || p->norm_weight),
                 DFLASH_ERR_ARG, "%s: null operand", who);
  DFLASH_REQUIRE(p->state_in != p->state_out, DFLASH_ERR_ARG, "%s: state_out must not alias state_in", who);
  auto ok = [](int dt) { return dt == DFLASH_BF16 || dt == DFLASH_FP16 || dt == DFLASH_FP32; };
  DFLASH_REQUIRE(ok(p->param_dtype) && ok(p->state_dtype) && (!p->z || ok(p->weight_dtype)), DFLASH_ERR_ARG, "%s: unknown dtype code", who);
  const int slots = p->slots, T = p->T, Hk = p->Hk, Hv = p->Hv, D = p->D;
  DFLASH_REQUIRE(slots >= 0 && T >= 1 && T <= 16 && Hk > 0 && Hv > 0 && Hv % Hk == 0 && (D == 64 || D == 128), DFLASH_ERR_SHAPE,
                 "%s: 1 to 16 steps of heads of 64 or 128, whole groups of value heads; got %d steps, %d and %d heads of %d", who, T, Hk,
                 Hv, D);
  DFLASH_REQUIRE(p->qkv_row < (1ll << 26), DFLASH_ERR_SHAPE, "%s: rows of %lld elements", who, p->qkv_row);
  DFLASH_REQUIRE((long long)slots * Hv * 8 < (1ll << 31) && (long long)slots * T * (2ll * Hk + Hv) * D < (1ll << 31), DFLASH_ERR_SHAPE,
                 "%s: too many (slot, head) pairs", who);
  uintptr_t strides = 0;
  for (long long v : {p->qkv_slot, p->qkv_row, p->a_slot, p->a_row, p->b_slot, p->b_row, p->z_slot, p->z_row})
    DFLASH_REQUIRE(v >= 0, DFLASH_ERR_SHAPE, "%s: negative stride", who);
  strides = (uintptr_t)(p->qkv_slot | p->qkv_row) * 2;
  DFLASH_REQUIRE((((uintptr_t)p->qkv | (uintptr_t)p->conv_state | (uintptr_t)p->conv_w | (uintptr_t)p->conv_next | (uintptr_t)p->k |
                   (uintptr_t)p->qkv_out | strides) % 8) == 0,
                 DFLASH_ERR_ARG, "%s: projections, conv arrays and k must be 8-byte aligned", who);
  DFLASH_REQUIRE((((uintptr_t)p->state_in | (uintptr_t)p->state_out | (uintptr_t)p->y | (uintptr_t)p->tape | (uintptr_t)p->z |
                   (uintptr_t)p->norm_weight | (p->z ? (uintptr_t)(p->z_slot | p->z_row) * 2 : 0)) % 16) == 0,
                 DFLASH_ERR_ARG, "%s: states, y, tape, z and the norm weight must be 16-byte aligned", who);
  if (slots == 0) return DFLASH_OK;

  GdnArgs a = {};
  a.state_in = p->state_in; a.state_out = p->state_out; a.y = p->y; a.tape = p->tape;
  a.T = T; a.Hk = Hk; a.Hv = Hv; a.Dk = a.Dv = D;
  a.heads = Divisor::of(Hv); a.group = Divisor::of(Hv / Hk); a.row_parts = Divisor::of(1);
  a.in_dtype = a.g_dtype = a.beta_dtype = DFLASH_BF16; a.state_dtype = p->state_dtype;
  a.z = p->z; a.z_batch = p->z_slot; a.z_row = p->z_row; a.norm_weight = p->norm_weight; a.weight_dtype = p->weight_dtype;
  a.eps = p->norm_eps;
  BlockArgs& b = a.block;
  b.qkv = (const uint16_t*)p->qkv; b.conv_state = (const uint16_t*)p->conv_state; b.conv_w = (const uint16_t*)p->conv_w;
  b.a = (const uint16_t*)p->a; b.b = (const uint16_t*)p->b; b.A_log = p->A_log; b.dt_bias = p->dt_bias;
  b.conv_next = (uint16_t*)p->conv_next; b.k_out = (uint16_t*)p->k; b.qkv_out = (uint16_t*)p->qkv_out; b.g_out = p->g;
  b.qkv_slot = p->qkv_slot; b.qkv_row = p->qkv_row; b.a_slot = p->a_slot; b.a_row = p->a_row; b.b_slot = p->b_slot; b.b_row = p->b_row;
  b.param_dt = p->param_dtype; b.eps = p->eps;
  const double inv_scale = 1.0 / sqrt((double)D);
  b.scale_q = as_bf16_scalar(inv_scale * inv_scale);
  b.scale_k = as_bf16_scalar(inv_scale);

  hipStream_t s = (hipStream_t)stream;
  void* args[] = {&a};
  if (D == 128 && p->state_dtype == DFLASH_FP32) {  // the closed form, its output norm in the same launch
    // A compute unit holds one workgroup of thirteen waves or two of four.  us for 16 tokens (one token), thirteen waves and four: 256 heads
    // 13.7 (13.3) and about 17 (15), 288 heads 24.3 (23.5) and 21.5 (19.7), 512 heads 25.7 (25.3) and 22.5 (19.7), 768 heads 38.0 (36.0) and
    // 35.8 (30.3), 1024 heads 50.1 (47.3) and 42.7 (35.8).
    const bool wide = slots * Hv <= qmm_stream_grid();
    const void* fn = wide ? (p->z ? (const void*)gdn_forward_chunk_128<false, true, true, kThirteenWaves>
                                : (const void*)gdn_forward_chunk_128<false, false, true, kThirteenWaves>)
                          : (p->z ? (const void*)gdn_forward_chunk_128<false, true, true, kFourWaves>
                                : (const void*)gdn_forward_chunk_128<false, false, true, kFourWaves>);
    DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)(slots * Hv)), dim3(wide ? kBlockThreads : kThreads), args, kChunkLdsFloats * sizeof(float), s));
    return DFLASH_OK;
  }
  int rows = D;
  const void* fn = forward_rows_for<true>(p->state_dtype, slots, Hv, D, D, &rows);
  a.row_parts = Divisor::of(D / rows);
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)(slots * Hv * (D / rows))), dim3(kThreads), args, 0, s));
  return p->z ? gdn_gated_norm_launch(p->y, p->z, p->norm_weight, p->y, slots, T, Hv, D, p->z_slot, p->z_row, DFLASH_BF16, p->weight_dtype,
                                      p->norm_eps, s)
              : DFLASH_OK;
}

extern "C" int dflash_gdn_forward_tape(const void* q, const void* k, const void* v, const void* g,
                                       const void* beta, const void* state_in, void* state_out,
                                       void* y, float* tape, const uint8_t* mask, int slots, int T,
                                       int Hk, int Hv, int Dk, int Dv, int in_dtype, int g_dtype,
                                       int beta_dtype, int state_dtype, int g_per_dk, void* stream) {
  return dflash::gdn_forward_launch("dflash_gdn_forward_tape", q, k, v, g, beta, state_in, state_out, y, tape, mask,
                                    nullptr, nullptr, DFLASH_FP32, 0.f, slots, T, Hk, Hv, Dk, Dv, in_dtype, g_dtype,
                                    beta_dtype, state_dtype, g_per_dk, stream);
}

extern "C" int dflash_gdn_forward_tape_norm(const void* q, const void* k, const void* v, const void* g,
                                            const void* beta, const void* state_in, void* state_out,
                                            const void* z, const void* norm_weight, void* out, float* tape,
                                            const uint8_t* mask, int slots, int T, int Hk, int Hv, int Dk, int Dv,
                                            int in_dtype, int g_dtype, int beta_dtype, int state_dtype,
                                            int weight_dtype, int g_per_dk, float eps, void* stream) {
  DFLASH_REQUIRE(z && norm_weight, DFLASH_ERR_ARG, "dflash_gdn_forward_tape_norm: null z or norm weight");
  return dflash::gdn_forward_launch("dflash_gdn_forward_tape_norm", q, k, v, g, beta, state_in, state_out, out, tape,
                                    mask, z, norm_weight, weight_dtype, eps, slots, T, Hk, Hv, Dk, Dv, in_dtype,
                                    g_dtype, beta_dtype, state_dtype, g_per_dk, stream);
}

extern "C" size_t dflash_gdn_forward_workspace_bytes(int slots, int T, int Hk, int Hv, int Dk, int Dv, int in_dtype, int g_per_dk) {
  using namespace dflash;
  return gdn_prompt_covers(slots, T, Hk, Hv, Dk, Dv, in_dtype, g_per_dk) ? gdn_prompt_workspace_bytes(slots, T, Hk, Hv, Dk) : 0;
}

extern "C" int dflash_gdn_forward(const void* q, const void* k, const void* v, const void* g, const void* beta,
                                  const void* state_in, void* state_out, const void* z, const void* norm_weight, void* y,
                                  float* tape, const uint8_t* mask, void* workspace, size_t workspace_bytes,
                                  long long z_batch_stride, long long z_row_stride, int slots, int T,
                                  int Hk, int Hv, int Dk, int Dv, int in_dtype, int g_dtype, int beta_dtype, int state_dtype,
                                  int weight_dtype, int g_per_dk, float eps, void* stream) {
  return dflash::gdn_forward_launch("dflash_gdn_forward", q, k, v, g, beta, state_in, state_out, y, tape, mask, z, norm_weight,
                                    weight_dtype, eps, slots, T, Hk, Hv, Dk, Dv, in_dtype, g_dtype, beta_dtype, state_dtype,
                                    g_per_dk, stream, workspace, workspace_bytes, z_batch_stride, z_row_stride);
}
