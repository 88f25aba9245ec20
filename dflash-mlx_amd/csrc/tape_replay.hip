// GatedDeltaNet tape replay for gfx950 (MI355X).
//
// Counterpart of the reference's `tape_replay{,_vec}{,_mask}` Metal kernels
// (dflash_mlx/kernels.py:227-325, dispatcher :361-407; array-op form :328-358):
// re-apply the first `steps` recorded (k_t, delta_t, g_t) updates to a recurrent
// state S[Dv][Dk] (Dk contiguous),
//     S[dv][dk] <- g_t * S[dv][dk] + k_t[dk] * delta_t[dv].
//
// The operation moves 2*Dv*Dk*4 bytes of state per head and almost nothing
// else, so it is laid out for HBM streaming:
//  * a workgroup has a head, or 32 or 64 rows of one; all of its part of the state
//    is in flight at once, in and out in full 128-byte lines;
//  * the tape (k, delta, g of <= T steps) is staged once into LDS as fp32;
//  * for an fp32 state the T sequential sweeps are folded into a single one,
//      S_a = (prod g) S0 + sum_t delta_t (x) (c_t k_t),  c_t = prod_{u>t} g_u
//    (c_t folded into the staged k rows, per-Dk gates included), in registers
//    (replay_rows) or, 128x128 heads with per-Dk gates, as a rank-16 update on the
//    fp32 matrix cores (replay_f32_128).  bf16/fp16 states, which the reference rounds after every step (kernels.py:281-283),
//    and callers that ask for it keep the step-by-step order (replay_rows, replay_generic);
//  * the accepted length is read per slot from device memory, so a rollback
//    does not need the host to know it, and one launch covers all layers.
#include "dflash_common.h"

namespace dflash {
namespace {

constexpr int kThreads = 256;

struct ReplayArgs {
  const void* tape;
  const void* k;
  const void* g;
  const void* state_in;
  void* state_out;
  const int32_t* steps_dev;
  const uint8_t* mask;
  int steps_host;
  int T, Hk, Hv, Dk, Dv;
  Divisor heads, group, row_parts;  // by Hv, by Hv / Hk, by the workgroups of a head (replay_rows)
  int state_dtype, tape_dtype, k_dtype, g_dtype, g_per_dk;
  // the conv window of the same layer, rebuilt by workgroups behind the replay's (none: conv_keep 0)
  const char* conv_prev;
  const char* conv_qkv;
  char* conv_out;
  size_t conv_row_bytes;
  int conv_keep, conv_vec16;
  int replay_blocks;  // workgroups of the replay itself
};

// LDS layout (floats): sA[Dv][T] (delta, t contiguous) | sK[T][Dk] | sG[T][Dk or 1] | sGt[Dk]
struct Smem {
  float* sA;
  float* sK;
  float* sG;
  float* sGt;
};

// `Tl` is the number of step slots the LDS tables hold (>= the steps staged).
__device__ __forceinline__ Smem carve(float* base, const ReplayArgs& a, int Tl) {
  Smem s;
  s.sA = base;
  s.sK = s.sA + (size_t)a.Dv * Tl;
  s.sG = s.sK + (size_t)Tl * a.Dk;
  s.sGt = s.sG + (size_t)Tl * (a.g_per_dk ? a.Dk : 1);
  return s;
}

// Stage the first `n` steps of this (slot, head) into LDS tables of `Tl` step
// slots.  Masked steps become delta = 0, k = 0, g = 1 (a no-op step) so later code
// need not look at the mask; step slots n..fill-1 are zero-filled (g = 1) as well.
__device__ __forceinline__ void stage_tape(const ReplayArgs& a, const Smem& s, int slot, int hv,
                                           int n, int Tl, int fill) {
  const int hk = hv / (a.Hv / a.Hk);
  const int tid = threadIdx.x;
  const size_t slotT = (size_t)slot * a.T;
  for (int i = tid; i < fill * a.Dv; i += kThreads) {
    const int t = i / a.Dv, dv = i - t * a.Dv;
    float d = 0.f;
    if (t < n && (a.mask == nullptr || a.mask[slotT + t] != 0)) {
      d = load_as_f32(a.tape, ((slotT + t) * a.Hv + hv) * a.Dv + dv, a.tape_dtype);
    }
    s.sA[(size_t)dv * Tl + t] = d;
  }
  for (int i = tid; i < fill * a.Dk; i += kThreads) {
    const int t = i / a.Dk, dk = i - t * a.Dk;
    const bool on = t < n && (a.mask == nullptr || a.mask[slotT + t] != 0);
    float kv = 0.f;
    if (on) kv = load_as_f32(a.k, ((slotT + t) * a.Hk + hk) * a.Dk + dk, a.k_dtype);
    s.sK[i] = kv;
    if (a.g_per_dk) {
      float gv = 1.f;
      if (on) gv = load_as_f32(a.g, ((slotT + t) * a.Hv + hv) * a.Dk + dk, a.g_dtype);
      s.sG[i] = gv;
    }
  }
  if (!a.g_per_dk) {
    for (int t = tid; t < fill; t += kThreads) {
      float gv = 1.f;
      if (t < n && (a.mask == nullptr || a.mask[slotT + t] != 0)) {
        gv = load_as_f32(a.g, (slotT + t) * a.Hv + hv, a.g_dtype);
      }
      s.sG[t] = gv;
    }
  }
}

// Fold the suffix products of g into the staged k rows; leave prod(g) in sGt.
__device__ __forceinline__ void fold_gates(const ReplayArgs& a, const Smem& s, int n) {
  for (int dk = threadIdx.x; dk < a.Dk; dk += kThreads) {
    float c = 1.f;
    for (int t = n - 1; t >= 0; --t) {
      s.sK[(size_t)t * a.Dk + dk] *= c;
      c *= a.g_per_dk ? s.sG[(size_t)t * a.Dk + dk] : s.sG[t];
    }
    s.sGt[dk] = c;
  }
}

__device__ __forceinline__ int slot_steps(const ReplayArgs& a, int slot) {
  int n = a.steps_dev ? a.steps_dev[slot] : a.steps_host;
  n = n < 0 ? 0 : n;
  return n > a.T ? a.T : n;
}

// Workgroups beyond the replay's own rebuild the conv window, one output row each.  True if this
// workgroup was one of them (and is done).
__device__ __forceinline__ bool conv_window_workgroup(const ReplayArgs& a, int block) {
  if (block < a.replay_blocks) return false;
  const int b = block - a.replay_blocks;
  const int slot = b / a.conv_keep, j = b % a.conv_keep;
  const int steps = a.steps_dev ? a.steps_dev[slot] : a.steps_host;
  if (a.conv_vec16) conv_rebuild_row<uint4>(a.conv_prev, a.conv_qkv, a.conv_out, steps, a.T, a.conv_keep, a.conv_row_bytes, slot, j);
  else conv_rebuild_row<unsigned char>(a.conv_prev, a.conv_qkv, a.conv_out, steps, a.T, a.conv_keep, a.conv_row_bytes, slot, j);
  return true;
}

// ---------------------------------------------------------------------------
// fp32 state, Dk = Dv = 128, T <= 16, a gate per element of a row: the folded sweep as a rank-16 update on the matrix cores.
//   S_out^T = diag(prod g) S_in^T + K'^T Delta,   K'[t][dk] = c_t[dk] k_t[dk]  (16 steps = 4 MFMAs
// of 16 x 16 x 4 fp32 per 16 x 16 tile).  The state sits in registers in accumulator layout
// (see swap_row_bit) and goes in and out in full 128-byte lines.
// LDS (floats): sK[16][kPad] | sD[16][kPad] | sG[16][128] | sGt[128]
// ---------------------------------------------------------------------------
constexpr int kPad = 132;  // row stride of the staged tables: step rows fall on different banks
constexpr size_t kReplayF32LdsFloats = 2 * 16 * kPad + 16 * 128 + 128;

// st (accumulator layout) <- diag(sGt) st + K'^T Delta over the first 4 NB steps; MFMA j of a tile
// covers steps 4 j + kq.
template <int NB>
__device__ __forceinline__ void rank_update(f32x4_t (&st)[2][8], const float* sK, const float* sD, const float* sGt,
                                            int wave, int li, int kq) {
  float dB[2][NB > 0 ? NB : 1];  // delta[step][32 wave + 16 t2 + li]
#pragma unroll
  for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
    for (int j = 0; j < NB; ++j) dB[t2][j] = sD[(4 * j + kq) * kPad + 32 * wave + 16 * t2 + li];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float kA[NB > 0 ? NB : 1];  // K'[step][16 c + li]
#pragma unroll
    for (int j = 0; j < NB; ++j) kA[j] = sK[(4 * j + kq) * kPad + 16 * c + li];
    const float4 gt4 = *reinterpret_cast<const float4*>(sGt + 16 * c + 4 * kq);
    const f32x4_t gt = {gt4.x, gt4.y, gt4.z, gt4.w};
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      f32x4_t acc = st[t2][c] * gt;
#pragma unroll
      for (int j = 0; j < NB; ++j) acc = mfma4(kA[j], dB[t2][j], acc);
      st[t2][c] = acc;
    }
  }
}

template <bool TAPE_WIDE, bool K_WIDE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3, 3))) void replay_f32_128(ReplayArgs a) {
  extern __shared__ float smem[];
  float* sK = smem;
  float* sD = sK + 16 * kPad;
  float* sG = sD + 16 * kPad;
  float* sGt = sG + 16 * 128;
  if (conv_window_workgroup(a, (int)blockIdx.x)) return;
  const int slot = a.heads.quotient((int)blockIdx.x), hv = (int)blockIdx.x - slot * a.Hv;
  const int n = slot_steps(a, slot);
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const f32x4_t* in = reinterpret_cast<const f32x4_t*>(a.state_in) + (size_t)blockIdx.x * (128 * 32);
  f32x4_t* out = reinterpret_cast<f32x4_t*>(a.state_out) + (size_t)blockIdx.x * (128 * 32);

  // The tape is asked for first and the state right behind it: loads return in issue order,
  // so the tape is in LDS and the gates are folded while the 64 KiB of state are still on
  // their way, instead of the state waiting in registers for the tape.  Every request goes out
  // before anything is awaited: thread (t = tid / 16, seg = tid % 16) fetches eight elements of
  // step t as raw bits, and what the bits mean (dtype, mask) is sorted out afterwards.
  // Rows are fetched whether accepted or not (every row below T exists): the accepted length
  // may itself still be on its way from device memory, and nothing here waits for it.
  const int t = tid >> 4, seg = tid & 15;
  const bool row = t < a.T;
  const bool g_wide = a.g_dtype == DFLASH_FP32;
  // raw bytes and bits in plain registers; nothing is computed from them until the state has
  // been asked for (see the fence below)
  u32x4_t rd0 = {0u, 0u, 0u, 0u}, rd1 = rd0, rk0 = rd0, rk1 = rd0, rg0 = rd0, rg1 = rd0;
  uint32_t mask_t = 1u;
  {
    const int hk = a.group.quotient(hv);
    const size_t slotT = (size_t)slot * a.T;
    if (row) {
      const size_t d_at = ((slotT + t) * a.Hv + hv) * 128 + 8 * seg;
      const size_t k_at = ((slotT + t) * a.Hk + hk) * 128 + 8 * seg;
      if (TAPE_WIDE) {
        rd0 = reinterpret_cast<const u32x4_t*>((const float*)a.tape + d_at)[0];
        rd1 = reinterpret_cast<const u32x4_t*>((const float*)a.tape + d_at)[1];
      } else {
        rd0 = *reinterpret_cast<const u32x4_t*>((const uint16_t*)a.tape + d_at);
      }
      if (K_WIDE) {
        rk0 = reinterpret_cast<const u32x4_t*>((const float*)a.k + k_at)[0];
        rk1 = reinterpret_cast<const u32x4_t*>((const float*)a.k + k_at)[1];
      } else {
        rk0 = *reinterpret_cast<const u32x4_t*>((const uint16_t*)a.k + k_at);
      }
      if (a.mask != nullptr) mask_t = a.mask[slotT + t];
      if (g_wide) {
        rg0 = reinterpret_cast<const u32x4_t*>((const float*)a.g + d_at)[0];
        rg1 = reinterpret_cast<const u32x4_t*>((const float*)a.g + d_at)[1];
      } else {
        rg0 = *reinterpret_cast<const u32x4_t*>((const uint16_t*)a.g + d_at);
      }
    }
  }

  f32x4_t st[2][8];
#pragma unroll
  for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
    for (int c = 0; c < 8; ++c) st[t2][c] = __builtin_nontemporal_load(&in[memory_index(wave, li, kq, t2, c)]);

  // Fence: the state's loads are out before any of the tape's values is looked at, so the
  // wait that the first use brings covers the tape only (loads return in issue order).
  asm volatile("" : "+v"(rd0), "+v"(rd1), "+v"(rk0), "+v"(rk1), "+v"(rg0), "+v"(rg1), "+v"(mask_t)::"memory");

  // masked and missing steps are (delta = 0, k = 0, g = 1): no-op steps
  {
    const bool keep = t < n && mask_t != 0;
    Raw8<TAPE_WIDE> rd;
    Raw8<K_WIDE> rk;
    const u32x4_t zero = {0u, 0u, 0u, 0u};
    auto as_uint4 = [](u32x4_t v) { return uint4{v.x, v.y, v.z, v.w}; };
    rd.w[0] = as_uint4(keep ? rd0 : zero);
    rd.w[TAPE_WIDE ? 1 : 0] = as_uint4(keep ? (TAPE_WIDE ? rd1 : rd0) : zero);
    rk.w[0] = as_uint4(keep ? rk0 : zero);
    rk.w[K_WIDE ? 1 : 0] = as_uint4(keep ? (K_WIDE ? rk1 : rk0) : zero);
    raw8_to_lds<TAPE_WIDE>(rd, a.tape_dtype, sD + t * kPad + 8 * seg);
    raw8_to_lds<K_WIDE>(rk, a.k_dtype, sK + t * kPad + 8 * seg);
    float* dst = sG + t * 128 + 8 * seg;
    if (!keep) {
      reinterpret_cast<float4*>(dst)[0] = reinterpret_cast<float4*>(dst)[1] = float4{1.f, 1.f, 1.f, 1.f};
    } else if (g_wide) {
      Raw8<true> rg;
      rg.w[0] = as_uint4(rg0), rg.w[1] = as_uint4(rg1);
      raw8_to_lds<true>(rg, a.g_dtype, dst);
    } else {
      Raw8<false> rg;
      rg.w[0] = as_uint4(rg0);
      raw8_to_lds<false>(rg, a.g_dtype, dst);
    }
  }
  __syncthreads();
  // suffix products of the gates into the k rows; their total into sGt
  if (tid < 128) {
    float c = 1.f;
    for (int t = n - 1; t >= 0; --t) {
      sK[t * kPad + tid] *= c;
      c *= sG[t * 128 + tid];
    }
    sGt[tid] = c;
  }
  __syncthreads();

#pragma unroll
  for (int m = 0; m < 4; ++m) {
    swap_row_bit(st[0][2 * m], st[0][2 * m + 1]);
    swap_row_bit(st[1][2 * m], st[1][2 * m + 1]);
  }
  // n is uniform over the workgroup: blocks of four steps beyond it are skipped
  switch ((n + 3) >> 2) {
    case 0: rank_update<0>(st, sK, sD, sGt, wave, li, kq); break;
    case 1: rank_update<1>(st, sK, sD, sGt, wave, li, kq); break;
    case 2: rank_update<2>(st, sK, sD, sGt, wave, li, kq); break;
    case 3: rank_update<3>(st, sK, sD, sGt, wave, li, kq); break;
    default: rank_update<4>(st, sK, sD, sGt, wave, li, kq); break;
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    swap_row_bit(st[0][2 * m], st[0][2 * m + 1]);
    swap_row_bit(st[1][2 * m], st[1][2 * m + 1]);
  }
#pragma unroll
  for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
    for (int c = 0; c < 8; ++c) __builtin_nontemporal_store(st[t2][c], &out[memory_index(wave, li, kq, t2, c)]);
}

// ---------------------------------------------------------------------------
// Dk = 64 or 128, T <= 16, one gate per head: a thread keeps 8 consecutive columns of R rows of S in registers from
// the first step to the last.  STATE = bf16 / fp16: step by step, rounded to that type after every step, three
// and a half vector instructions per element and step (unpack, product, fma, half a conversion of two).  STATE =
// fp32: the folded single sweep.  Each wave multiplies the gates up by itself, out of the lanes that fetched them, and k is
// scaled on its way to LDS: with the products made there, one dependent read per step, and a barrier, 32 heads took 6.0 us.
//  * One request of 16 bytes per row and lane; the tape is asked for first, the state right behind it, and nothing
//    is looked at before all of it is on its way (see replay_f32_128).
//  * k of a step is read from LDS once for the R rows; a wave's reads of it are 512 consecutive bytes.
//  * Bound by its vector instructions: 128 x 128 at 16 steps are 3.6 k of them per wave of a head that one workgroup
//    computes, so a launch of few heads is spread over 32 rows per workgroup (R = 2, 64 x 64 heads: R = 1).
// Measured against replay_generic, which served these before (one workgroup per head, 2-byte accesses, a division
// per element), bf16 states, 16 / 6 steps, us: 32 heads of 128 x 128 97.8 / 45.6 -> 5.1 / 3.9, 1536 heads 148 / 69 -> 44 / 21;
// 32 heads of 64 x 64 26.6 / 13.4 -> 4.0 / 3.2, 1536 heads 39 / 21 -> 12.3 / 7.9.  fp32 states of 128 x 128 against a rank-16 update on
// the fp32 matrix cores, a workgroup per head (the form replay_f32_128 keeps for gates per element; same bits): 1 head 6.7 / 6.2 -> 4.0 / 3.5,
// 32 heads 7.4 / 6.8 -> 4.4 / 3.9, 192 heads 8.3 / 7.4 -> 6.9 / 6.3, 1536 heads 40.9 / 39.7 -> 37.2 / 35.7 (5.7 TB/s); of 64 x 64, 32 heads
// 4.7 / 3.9 -> 3.5 / 3.2, 1536 heads 14.5 / 13.1 -> 11.8 / 11.6.
// ---------------------------------------------------------------------------
template <int STATE, int DK, int R>
__device__ __forceinline__ void replay_rows_of(const ReplayArgs& a, int block) {
  constexpr bool kWide = STATE == DFLASH_FP32;
  constexpr int kLanes = DK / 8, kPass = kThreads / kLanes, kRows = kPass * R;  // lanes of a row, rows of a pass, of the workgroup
  constexpr int kD = kRows / 16, kK = DK / 16;  // elements of delta and k that a thread brings
  __shared__ __align__(16) float sK[16 * DK];
  __shared__ __align__(16) float sD[16 * kRows];
  __shared__ float sG[16];
  if (conv_window_workgroup(a, block)) return;
  const int head = a.row_parts.quotient(block), row0 = (block - head * (int)a.row_parts.by) * kRows;
  const int slot = a.heads.quotient(head), hv = head - slot * a.Hv, hk = a.group.quotient(hv);
  const int n = slot_steps(a, slot);
  const int tid = threadIdx.x, t = tid >> 4, seg = tid & 15;
  const size_t slotT = (size_t)slot * a.T;

  // (every row below T exists, accepted or not)
  uint32_t rd[kD] = {}, rk[kK] = {}, mask_t = 1u, mask_g = 1u, g_bits = 0u;
  if (t < a.T) {
    load_bits<kD>(a.tape, ((slotT + t) * a.Hv + hv) * a.Dv + row0 + kD * seg, a.tape_dtype == DFLASH_FP32, rd);
    load_bits<kK>(a.k, ((slotT + t) * a.Hk + hk) * DK + kK * seg, a.k_dtype == DFLASH_FP32, rk);
    if (a.mask != nullptr) mask_t = a.mask[slotT + t];
  }
  // thread t < 16 also fetches the gate of step t; fp32 states: lanes t, 16 + t, .. of every wave
  const int gt = kWide ? tid & 15 : tid;
  if (gt < a.T) {
    const size_t at = (slotT + gt) * a.Hv + hv;
    if (a.g_dtype == DFLASH_FP32) g_bits = ((const uint32_t*)a.g)[at];
    else g_bits = ((const uint16_t*)a.g)[at];
    if (a.mask != nullptr) mask_g = a.mask[slotT + gt];
  }
  const int rr = tid / kLanes, c8 = tid % kLanes;
  // fp32: a lane's columns are four of either half of the row, so that every access of a row is in one piece
  const size_t at0 = ((size_t)head * a.Dv + row0 + rr) * DK + (kWide ? 4 : 8) * c8;
  u32x4_t raw[R][kWide ? 2 : 1];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const size_t at = at0 + (size_t)i * kPass * DK;
    if (kWide) {
      const u32x4_t* src = reinterpret_cast<const u32x4_t*>((const float*)a.state_in + at);
      raw[i][0] = __builtin_nontemporal_load(src);
      raw[i][kWide ? 1 : 0] = __builtin_nontemporal_load(src + DK / 8);
    } else {
      raw[i][0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>((const uint16_t*)a.state_in + at));
    }
  }
#pragma unroll
  for (int e = 0; e < kD; ++e) asm volatile("" : "+v"(rd[e])::"memory");
#pragma unroll
  for (int e = 0; e < kK; ++e) asm volatile("" : "+v"(rk[e])::"memory");
  asm volatile("" : "+v"(mask_t), "+v"(mask_g), "+v"(g_bits)::"memory");

  // masked and missing steps are (delta = 0, k = 0, g = 1): no-op steps
  const uint32_t g_word[1] = {g_bits};
  const float gate = gt < n && mask_g != 0 ? bits_element(g_word, 0, a.g_dtype) : 1.f;
  float total = 1.f, after = 1.f;  // products of all gates and of those behind step t, which goes into k
  if (kWide) {
#pragma unroll
    for (int s = 15; s >= 0; --s) {
      after = t == s ? total : after;
      total *= __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(gate), s));
    }
  } else if (tid < 16) {
    sG[tid] = gate;
  }
  const bool keep = t < n && mask_t != 0;
#pragma unroll
  for (int e = 0; e < kD; ++e) sD[t * kRows + kD * seg + e] = keep ? bits_element(rd, e, a.tape_dtype) : 0.f;
#pragma unroll
  for (int e = 0; e < kK; ++e) sK[t * DK + (kWide ? kK * seg + e : plane_index<DK>(kK * seg + e))] = keep ? bits_element(rk, e, a.k_dtype) * after : 0.f;
  __syncthreads();

  if constexpr (kWide) {
    float v[R][8];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] = __uint_as_float(raw[i][kWide ? e >> 2 : 0][e & 3]) * total;
    for (int s0 = 0; s0 < n; s0 += 4) {  // (steps from n on are no-op steps)
#pragma unroll
      for (int s = s0; s < s0 + 4; ++s) {
        float k8[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float4 k4 = *reinterpret_cast<const float4*>(sK + s * DK + h * (DK / 2) + 4 * c8);
          k8[4 * h] = k4.x, k8[4 * h + 1] = k4.y, k8[4 * h + 2] = k4.z, k8[4 * h + 3] = k4.w;
        }
#pragma unroll
        for (int i = 0; i < R; ++i) {
          const float d = sD[s * kRows + i * kPass + rr];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[i][e] = fmaf(d, k8[e], v[i][e]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[i][kWide ? e >> 2 : 0][e & 3] = __float_as_uint(v[i][e]);
  } else {
#pragma unroll 2
    for (int s = 0; s < n; ++s) {
      float k8[8];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float4 k4 = *reinterpret_cast<const float4*>(sK + s * DK + h * (DK / 2) + 4 * c8);
        k8[4 * h] = k4.x, k8[4 * h + 1] = k4.y, k8[4 * h + 2] = k4.z, k8[4 * h + 3] = k4.w;
      }
      const float g = sG[s];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float d = sD[s * kRows + i * kPass + rr];
#pragma unroll
        for (int p = 0; p < 4; ++p)
          raw[i][0][p] = pack_pair<STATE>(fmaf(pair_lo<STATE>(raw[i][0][p]), g, k8[2 * p] * d),
                                          fmaf(pair_hi<STATE>(raw[i][0][p]), g, k8[2 * p + 1] * d));
      }
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const size_t at = at0 + (size_t)i * kPass * DK;
    if (kWide) {
      u32x4_t* dst = reinterpret_cast<u32x4_t*>((float*)a.state_out + at);
      __builtin_nontemporal_store(raw[i][0], dst);
      __builtin_nontemporal_store(raw[i][kWide ? 1 : 0], dst + DK / 8);
    } else {
      __builtin_nontemporal_store(raw[i][0], reinterpret_cast<u32x4_t*>((uint16_t*)a.state_out + at));
    }
  }
}

template <int STATE, int DK, int R>
__global__ __launch_bounds__(kThreads) void replay_rows(ReplayArgs a) {
  replay_rows_of<STATE, DK, R>(a, (int)blockIdx.x);
}

// Layers that hold tensors of their own, of one shape, in one launch: a workgroup finds its layer by its place and the layer's
// addresses among the arguments.  A launch per layer leaves most of the chip idle for its 5 to 6 us and costs the host 4.  Kernel
// time, a launch each and together: 20 layers of 2 x 32 heads of 128 x 128, bf16 states, 13 steps 119 -> 36 us; 10 of 64 heads, fp32,
// 8 steps 50 -> 18; 48 of 32 heads, fp32, 7 steps 228 -> 42 (two launches).  The calls around them 188 -> 106, 89 -> 56 and
// 430 -> 254 us: what is left is the host's, two allocations a layer and the caches' own steps.
constexpr int kLayersAtOnce = 32;  // their addresses and the rest of the arguments are 2.3 KB
struct LayersArgs {
  ReplayArgs one;  // of a layer, without addresses
  Divisor per_layer, windows;  // by the workgroups of a layer that replay and that rebuild its conv window
  int replay_blocks;  // of all layers
  dflash_rollback_operands at[kLayersAtOnce];
};

template <int STATE, int DK, int R>
__global__ __launch_bounds__(kThreads) void replay_rows_layers(LayersArgs p) {
  ReplayArgs a = p.one;
  int block = (int)blockIdx.x, layer;
  if (block < p.replay_blocks) {
    layer = p.per_layer.quotient(block);
    block -= layer * a.replay_blocks;
  } else {
    block -= p.replay_blocks;
    layer = p.windows.quotient(block);
    block += a.replay_blocks - layer * (int)p.windows.by;
  }
  const dflash_rollback_operands& at = p.at[layer];
  a.tape = at.tape, a.k = at.k, a.g = at.g, a.state_in = at.state_in, a.state_out = at.state_out;
  a.conv_prev = (const char*)at.conv_prev, a.conv_qkv = (const char*)at.qkv, a.conv_out = (char*)at.conv_out;
  replay_rows_of<STATE, DK, R>(a, block);
}

// The form of replay_rows for a head size and state type; rows: how many a workgroup computes.  heads: of all slots.  The lines
// of the fp32 states (16 bf16 steps, us with one / two / four / eight rows of a pass): 128 x 128, 32 heads 4.5 / 4.4 / 5.1 / 7.2,
// 192 heads 8.9 / 6.9 / 7.3 / 8.6, 256 heads 11.0 / 7.9 / 7.9 / 9.7, 384 heads 14.9 / 11.6 / 9.8 / 11.2, 1536 heads 42.6 / 39.5 / 37.2 / 39.9;
// eight rows also where they are one round of the chip and four rows a second one (two and three such workgroups fit a compute unit): 416 heads
// 15.9 / 13.6 / 13.3 / 11.4, 512 heads 17.6 / 15.4 / 14.3 / 12.8, 544 heads 18.6 / 16.2 / 15.7 / 17.1 (fp32 tapes, four and eight rows: 416 heads
// 13.5 / 12.0, 512 heads 14.6 / 13.7; a head per workgroup on the matrix cores 13.0 and 13.7).
// 64 x 64, 32 heads 3.5 / 4.0, 96 heads 4.1 / 4.2, 256 heads 5.1 / 4.5, 1536 heads 13.8 / 11.8.  Of the 16-bit ones: a whole head per
// workgroup from 1024 heads on, where k is staged once for more rows, but at 16 steps fewer waves cover each other's waits (128 x 128, 16 / 6
// steps, us, split and whole: 512 heads 16.0 / 10.0 and 19.3 / 10.3, 1024 heads 28.6 / 16.8 and 31.9 / 15.4, 1536 heads 41.6 / 25.4
// and 44.4 / 20.5; 64 x 64 at 1024 heads 10.6 / 7.2 and 9.6 / 6.1).
template <int STATE>
const void* replay_rows_for(int Dk, int Dv, long long heads, bool layers, int* rows) {
#define DFLASH_REPLAY_ROWS(DK_, R_, ROWS_) \
  return *rows = ROWS_, layers ? (const void*)replay_rows_layers<STATE, DK_, R_> : (const void*)replay_rows<STATE, DK_, R_>
  constexpr bool kWide = STATE == DFLASH_FP32;
  const bool many = kWide ? heads > (Dk == 128 ? 192 : 96) : heads >= 1024;
  constexpr int kMany = kWide ? 4 : 8;
  if (kWide && Dk == 128 && Dv % 128 == 0 && heads * (Dv / 64) > 3 * 256 && heads * (Dv / 128) <= 2 * 256) DFLASH_REPLAY_ROWS(128, 8, 128);
  if (Dk == 128 && many && Dv % (16 * kMany) == 0) DFLASH_REPLAY_ROWS(128, kMany, 16 * kMany);
  if (Dk == 128 && Dv % 32 == 0) DFLASH_REPLAY_ROWS(128, 2, 32);
  if (Dk == 64 && many && Dv % 64 == 0) DFLASH_REPLAY_ROWS(64, 2, 64);
  if (Dk == 64 && Dv % 32 == 0) DFLASH_REPLAY_ROWS(64, 1, 32);
  return nullptr;
#undef DFLASH_REPLAY_ROWS
}
const void* replay_rows_for(int state_dtype, int Dk, int Dv, long long heads, bool layers, int* rows) {
  return state_dtype == DFLASH_BF16   ? replay_rows_for<DFLASH_BF16>(Dk, Dv, heads, layers, rows)
         : state_dtype == DFLASH_FP16 ? replay_rows_for<DFLASH_FP16>(Dk, Dv, heads, layers, rows)
                                      : replay_rows_for<DFLASH_FP32>(Dk, Dv, heads, layers, rows);
}

// ---------------------------------------------------------------------------
// Generic shapes / dtypes.  EXACT = step-by-step order with a round-trip through
// the state dtype after every step; otherwise the folded single sweep (fp32 state).
// ---------------------------------------------------------------------------
template <bool EXACT>
__global__ __launch_bounds__(kThreads) void replay_generic(ReplayArgs a) {
  extern __shared__ float smem[];
  if (conv_window_workgroup(a, (int)blockIdx.x)) return;
  const Smem s = carve(smem, a, a.T);
  const int slot = blockIdx.x / a.Hv, hv = blockIdx.x % a.Hv;
  const int n = slot_steps(a, slot);
  const int dk4n = a.Dk >> 2;
  const size_t base = (size_t)blockIdx.x * a.Dv * a.Dk;

  stage_tape(a, s, slot, hv, n, a.T, n);
  __syncthreads();
  if (!EXACT) {
    fold_gates(a, s, n);
    __syncthreads();
  }

  for (int e = threadIdx.x; e < a.Dv * dk4n; e += kThreads) {
    const int dv = e / dk4n, c4 = e - dv * dk4n;
    const size_t off = base + (size_t)dv * a.Dk + 4 * c4;
    float v[4];
    if (a.state_dtype == DFLASH_FP32) {
      const float4 q = *reinterpret_cast<const float4*>((const float*)a.state_in + off);
      v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = load_as_f32(a.state_in, off + j, a.state_dtype);
    }
    const float* dl = s.sA + (size_t)dv * a.T;
    if (EXACT) {
      // masked steps were staged as (delta=0, k=0, g=1): s*1 + 0*0 keeps s bit-for-bit
      for (int t = 0; t < n; ++t) {
        const float d = dl[t];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float gv = a.g_per_dk ? s.sG[(size_t)t * a.Dk + 4 * c4 + j] : s.sG[t];
          float sv = v[j] * gv;
          sv = sv + s.sK[(size_t)t * a.Dk + 4 * c4 + j] * d;
          v[j] = round_through(sv, a.state_dtype);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] *= s.sGt[4 * c4 + j];
      for (int t = 0; t < n; ++t) {
        const float d = dl[t];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += d * s.sK[(size_t)t * a.Dk + 4 * c4 + j];
      }
    }
    if (a.state_dtype == DFLASH_FP32) {
      *reinterpret_cast<float4*>((float*)a.state_out + off) = make_float4(v[0], v[1], v[2], v[3]);
    } else if (a.state_dtype == DFLASH_BF16) {
#pragma unroll
      for (int j = 0; j < 4; ++j) ((uint16_t*)a.state_out)[off + j] = (uint16_t)f32_to_bf16_bits(v[j]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) ((uint16_t*)a.state_out)[off + j] = (uint16_t)f32_to_f16_bits(v[j]);
    }
  }
}

bool valid_dtype(int dt) { return dt == DFLASH_BF16 || dt == DFLASH_FP16 || dt == DFLASH_FP32; }

}  // namespace
}  // namespace dflash

namespace dflash {
namespace {
// The replay launch; with qkv != nullptr the conv window of the same slots rides along
// (conv_prev [slots, keep, C] or NULL, qkv [slots, T, C], conv_out [slots, keep, C]).
int replay_launch(const void* tape, const void* k, const void* g, const void* state_in, void* state_out,
                  const int32_t* steps_dev, int steps_host, const uint8_t* mask, int slots, int T, int Hk,
                  int Hv, int Dk, int Dv, int state_dtype, int tape_dtype, int k_dtype, int g_dtype,
                  int g_per_dk, int exact_order, const void* conv_prev, const void* qkv, void* conv_out,
                  int keep, int C, int qkv_elem_bytes, void* stream) {
  DFLASH_REQUIRE(state_in && state_out, DFLASH_ERR_ARG, "dflash_tape_replay: null state");
  DFLASH_REQUIRE(state_in != state_out, DFLASH_ERR_ARG,
                 "dflash_tape_replay: state_out must not alias state_in");
  DFLASH_REQUIRE(valid_dtype(state_dtype) && valid_dtype(tape_dtype) && valid_dtype(k_dtype) &&
                     valid_dtype(g_dtype),
                 DFLASH_ERR_ARG, "dflash_tape_replay: unknown dtype code");
  DFLASH_REQUIRE(slots >= 0 && T >= 0 && Hk > 0 && Hv > 0 && Dk > 0 && Dv > 0, DFLASH_ERR_SHAPE,
                 "dflash_tape_replay: non-positive dimension");
  DFLASH_REQUIRE(Hv % Hk == 0, DFLASH_ERR_SHAPE,
                 "dflash_tape_replay: cannot align K heads %d to tape heads %d", Hk, Hv);
  DFLASH_REQUIRE(Dk % 4 == 0 && Dk <= 1024, DFLASH_ERR_SHAPE,
                 "dflash_tape_replay: Dk=%d must be a multiple of 4 and <= 1024", Dk);
  DFLASH_REQUIRE(T == 0 || (tape && k && g), DFLASH_ERR_ARG, "dflash_tape_replay: null tape");
  if (slots == 0) return DFLASH_OK;
  const bool exact = exact_order != 0 || state_dtype != DFLASH_FP32;
  // the 128 x 128 kernel fetches tape, k and per-element gates 16 bytes at a time
  const bool aligned16 = (((uintptr_t)tape | (uintptr_t)k | (g_per_dk ? (uintptr_t)g : 0)) % 16) == 0;
  // one gate per head, at least a step: step by step for 16-bit states, folded for fp32 ones
  const void* by_rows = nullptr;
  int rows = Dv;
  if (!g_per_dk && T >= 1 && T <= 16 && aligned16 && (((uintptr_t)state_in | (uintptr_t)state_out) % 16) == 0 &&
      (!exact || state_dtype != DFLASH_FP32)) {
    const long long heads = (long long)slots * Hv;
    by_rows = replay_rows_for(state_dtype, Dk, Dv, heads, false, &rows);
  }
  // gates per element of a row: the matrix-core form
  const bool fast = !exact && g_per_dk && Dk == 128 && Dv == 128 && T <= 16 && aligned16;
  const size_t Tl = fast ? 16 : (size_t)T;
  const size_t smem_floats = by_rows ? 0
                             : fast  ? kReplayF32LdsFloats
                                     : (size_t)Dv * Tl + Tl * Dk + Tl * (g_per_dk ? Dk : 1) + (size_t)Dk;
  const size_t smem = smem_floats * sizeof(float);
  DFLASH_REQUIRE(state_dtype != DFLASH_FP32 ||
                     (((uintptr_t)state_in % 16) == 0 && ((uintptr_t)state_out % 16) == 0),
                 DFLASH_ERR_ARG, "dflash_tape_replay: fp32 state must be 16-byte aligned");
  DFLASH_REQUIRE(smem <= 64 * 1024, DFLASH_ERR_SHAPE,
                 "dflash_tape_replay: tape of T=%d steps needs %zu bytes of LDS (> 64 KiB)", T,
                 smem);
  DFLASH_REQUIRE((long long)slots * Hv < (1ll << 31), DFLASH_ERR_SHAPE,
                 "dflash_tape_replay: too many (slot, head) pairs");

  ReplayArgs a;
  a.tape = tape; a.k = k; a.g = g; a.state_in = state_in; a.state_out = state_out;
  a.steps_dev = steps_dev; a.mask = mask; a.steps_host = steps_host;
  a.T = T; a.Hk = Hk; a.Hv = Hv; a.Dk = Dk; a.Dv = Dv;
  a.heads = Divisor::of(Hv); a.group = Divisor::of(Hv / Hk); a.row_parts = Divisor::of(by_rows ? Dv / rows : 1);
  a.state_dtype = state_dtype; a.tape_dtype = tape_dtype; a.k_dtype = k_dtype;
  a.g_dtype = g_dtype; a.g_per_dk = g_per_dk ? 1 : 0;
  const long long blocks = (long long)slots * Hv * (by_rows ? Dv / rows : 1);
  DFLASH_REQUIRE(blocks < (1ll << 31), DFLASH_ERR_SHAPE, "dflash_tape_replay: too many workgroups");
  a.replay_blocks = (int)blocks;
  a.conv_prev = a.conv_qkv = nullptr; a.conv_out = nullptr; a.conv_row_bytes = 0; a.conv_keep = a.conv_vec16 = 0;
  long long conv_blocks = 0;
  if (qkv != nullptr) {
    DFLASH_REQUIRE(conv_out && conv_out != conv_prev, DFLASH_ERR_ARG,
                   "dflash_rollback_layer: conv_out must be given and must not alias conv_prev");
    DFLASH_REQUIRE(T > 0 && keep > 0 && C > 0 && qkv_elem_bytes > 0, DFLASH_ERR_SHAPE,
                   "dflash_rollback_layer: non-positive dimension of the conv window");
    a.conv_prev = (const char*)conv_prev; a.conv_qkv = (const char*)qkv; a.conv_out = (char*)conv_out;
    a.conv_row_bytes = (size_t)C * qkv_elem_bytes;
    a.conv_keep = keep;
    a.conv_vec16 = a.conv_row_bytes % 16 == 0 && (uintptr_t)qkv % 16 == 0 && (uintptr_t)conv_out % 16 == 0 &&
                   (uintptr_t)conv_prev % 16 == 0;
    conv_blocks = (long long)slots * keep;
    DFLASH_REQUIRE(blocks + conv_blocks < (1ll << 31), DFLASH_ERR_SHAPE,
                   "dflash_rollback_layer: too many workgroups");
  }

  const dim3 grid((unsigned)(blocks + conv_blocks)), block(kThreads);
  hipStream_t s = (hipStream_t)stream;
  if (by_rows != nullptr) {
    void* args[] = {&a};
    DFLASH_HIP_OK(hipLaunchKernel(by_rows, grid, block, args, 0, s));
    return DFLASH_OK;
  }
  if (exact) {
    hipLaunchKernelGGL(replay_generic<true>, grid, block, smem, s, a);
  } else if (fast) {
    const bool tw = tape_dtype == DFLASH_FP32, kw = k_dtype == DFLASH_FP32;
    if (tw && kw) hipLaunchKernelGGL((replay_f32_128<true, true>), grid, block, smem, s, a);
    else if (tw) hipLaunchKernelGGL((replay_f32_128<true, false>), grid, block, smem, s, a);
    else if (kw) hipLaunchKernelGGL((replay_f32_128<false, true>), grid, block, smem, s, a);
    else hipLaunchKernelGGL((replay_f32_128<false, false>), grid, block, smem, s, a);
  } else {
    hipLaunchKernelGGL(replay_generic<false>, grid, block, smem, s, a);
  }
  DFLASH_HIP_OK(hipGetLastError());
  return DFLASH_OK;
}
}  // namespace
}  // namespace dflash

extern "C" int dflash_tape_replay(const void* tape, const void* k, const void* g,
                                  const void* state_in, void* state_out, const int32_t* steps_dev,
                                  int steps_host, const uint8_t* mask, int slots, int T, int Hk,
                                  int Hv, int Dk, int Dv, int state_dtype, int tape_dtype,
                                  int k_dtype, int g_dtype, int g_per_dk, int exact_order,
                                  void* stream) {
  return dflash::replay_launch(tape, k, g, state_in, state_out, steps_dev, steps_host, mask, slots, T, Hk, Hv, Dk,
                               Dv, state_dtype, tape_dtype, k_dtype, g_dtype, g_per_dk, exact_order, nullptr,
                               nullptr, nullptr, 0, 0, 0, stream);
}

extern "C" int dflash_rollback_layer(const void* tape, const void* k, const void* g, const void* state_in,
                                     void* state_out, const void* conv_prev, const void* qkv, void* conv_out,
                                     const int32_t* steps_dev, int steps_host, int slots, int T, int Hk,
                                     int Hv, int Dk, int Dv, int state_dtype, int tape_dtype, int k_dtype,
                                     int g_dtype, int g_per_dk, int exact_order, int keep, int C,
                                     int qkv_elem_bytes, void* stream) {
  const bool window = qkv != nullptr && keep > 0;
  return dflash::replay_launch(tape, k, g, state_in, state_out, steps_dev, steps_host, nullptr, slots, T, Hk, Hv, Dk,
                               Dv, state_dtype, tape_dtype, k_dtype, g_dtype, g_per_dk, exact_order,
                               window ? conv_prev : nullptr, window ? qkv : nullptr, window ? conv_out : nullptr,
                               window ? keep : 0, window ? C : 0, window ? qkv_elem_bytes : 0, stream);
}

extern "C" int dflash_rollback_layers(const dflash_rollback_operands* layers, int count, int steps, int slots, int T, int Hk, int Hv,
                                      int Dk, int Dv, int state_dtype, int tape_dtype, int k_dtype, int g_dtype, int exact_order,
                                      int keep, int C, int qkv_elem_bytes, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(count == 0 || layers, DFLASH_ERR_ARG, "dflash_rollback_layers: null operands");
  DFLASH_REQUIRE(count >= 0 && slots >= 0 && T >= 0 && Hk > 0 && Hv > 0 && Dk > 0 && Dv > 0, DFLASH_ERR_SHAPE,
                 "dflash_rollback_layers: non-positive dimension");
  DFLASH_REQUIRE(valid_dtype(state_dtype) && valid_dtype(tape_dtype) && valid_dtype(k_dtype) && valid_dtype(g_dtype), DFLASH_ERR_ARG,
                 "dflash_rollback_layers: unknown dtype code");
  bool joint = count > 1 && slots > 0 && T >= 1 && T <= 16 && Hv % Hk == 0 && (state_dtype != DFLASH_FP32 || exact_order == 0);
  const bool window = keep > 0;
  const size_t row_bytes = window && C > 0 && qkv_elem_bytes > 0 ? (size_t)C * qkv_elem_bytes : 0;
  joint = joint && (!window || row_bytes != 0);
  bool vec16 = row_bytes % 16 == 0;
  for (int i = 0; i < count; ++i) {
    const dflash_rollback_operands& at = layers[i];
    const uintptr_t wide = (uintptr_t)at.tape | (uintptr_t)at.k | (uintptr_t)at.state_in | (uintptr_t)at.state_out;
    joint = joint && at.tape && at.k && at.g && at.state_in && at.state_out && at.state_in != at.state_out && wide % 16 == 0 &&
            (!window || (at.qkv && at.conv_out && at.conv_out != at.conv_prev));
    vec16 = vec16 && ((uintptr_t)at.conv_prev | (uintptr_t)at.qkv | (uintptr_t)at.conv_out) % 16 == 0;
  }
  for (int first = 0; first < count;) {
    const int here = count - first < kLayersAtOnce ? count - first : kLayersAtOnce;
    int rows = 0;
    const long long heads = (long long)slots * Hv;
    const void* const fn = joint && here > 1 ? replay_rows_for(state_dtype, Dk, Dv, heads * here, true, &rows) : nullptr;
    const long long blocks = fn ? heads * (Dv / rows) : 0, windows = window ? (long long)slots * keep : 0;
    if (fn == nullptr || (blocks + windows) * here >= (1ll << 31)) {
      // layer by layer, also for whatever that call refuses
      for (int i = first; i < first + here; ++i) {
        const dflash_rollback_operands& at = layers[i];
        const int rc = dflash_rollback_layer(at.tape, at.k, at.g, at.state_in, at.state_out, at.conv_prev, at.qkv, at.conv_out, nullptr,
                                             steps, slots, T, Hk, Hv, Dk, Dv, state_dtype, tape_dtype, k_dtype, g_dtype, 0, exact_order,
                                             keep, C, qkv_elem_bytes, stream);
        if (rc != DFLASH_OK) return rc;
      }
      first += here;
      continue;
    }
    LayersArgs p = {};
    ReplayArgs& a = p.one;
    a.steps_host = steps;
    a.T = T; a.Hk = Hk; a.Hv = Hv; a.Dk = Dk; a.Dv = Dv;
    a.heads = Divisor::of(Hv); a.group = Divisor::of(Hv / Hk); a.row_parts = Divisor::of(Dv / rows);
    a.state_dtype = state_dtype; a.tape_dtype = tape_dtype; a.k_dtype = k_dtype; a.g_dtype = g_dtype;
    a.conv_row_bytes = row_bytes; a.conv_keep = window ? keep : 0; a.conv_vec16 = vec16;
    a.replay_blocks = (int)blocks;
    p.per_layer = Divisor::of(blocks); p.windows = Divisor::of(windows > 0 ? windows : 1);
    p.replay_blocks = (int)(blocks * here);
    for (int i = 0; i < here; ++i) p.at[i] = layers[first + i];
    void* args[] = {&p};
    DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)((blocks + windows) * here)), dim3(kThreads), args, 0, (hipStream_t)stream));
    first += here;
  }
  return DFLASH_OK;
}
