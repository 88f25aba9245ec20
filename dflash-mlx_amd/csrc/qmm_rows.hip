// 4-bit affine matmul for any number of rows, y[M,N] = x[M,K] . round(s*q + b)^T (gfx950): prompts,
// and every other call the 16-row kernels do not serve.
//
// What the reference leaves to mx.quantized_matmul (dflash_mlx/verify_qmm.py:277-280).  A weight is
// dequantised to the activation type as the array-op form of this package does it (s*q + b in
// fp32, rounded once) and multiplied on the matrix cores with fp32 accumulation.
//
//  * A wave owns whole columns: a workgroup is 4 waves side by side, each 16*NT columns wide and all
//    16*MT rows high, so that a weight is dequantised once per 16*MT rows.  With KG = 2 a second
//    set of four waves takes the other half of every stage of K and the two halves meet in LDS
//    at the end: two waves per SIMD, so that one dequantises while the other multiplies, without
//    cutting the result any smaller.
//  * Codes, scales and x all go through LDS.  Read by the lanes that multiply them, neighbouring lanes would
//    ask for different rows, and a load that touches 16 or 64 rows costs the address unit 64 cycles
//    instead of 16: that, not arithmetic, bounded the form of this kernel that kept codes in
//    registers (4 + 8 such loads per 64 k and wave, 3072 cycles of address work per 1024 cycles of
//    matrix work).  Loads go to registers at the start of a stage and to the other LDS buffer at its end.
//  * dequantisation: code q sits in the low bits of a half word; as an fp16 subnormal that half is
//    q 2^-24, so fma_mix(half, s 2^24, b) is s q + b in one instruction and exact up to its one
//    rounding; the conversion to the activation type packs two at a time: 19 vector instructions per
//    8 weights, 60 % of the matrix instructions' time at MT = 8.
//  * W is the A operand (rows of the tile = columns of y), x the B operand, and the columns of a
//    wave are dealt to its tiles so that a lane ends up with 4*NT consecutive columns of one row.
//  * Where the tiles do not fill the chip, K is cut into slices: workgroups leave fp32 partial tiles in
//    the workspace, and whoever arrives last at a tile adds them in order of k.  Nobody waits.  Deterministic.
//    Of more tiles than the chip takes at once, only those of the last, incomplete round are cut: 1088 tiles of
//    5120 x 34816 are 4 rounds and a quarter instead of 5 (a 27B layer over 1024 tokens 787 -> 758 us).
//
// Measured (kernel time, group 64, before that cut): 1024 rows of 5120 x 34816 415 us (880 TFLOP/s; torch's bf16 product of weights
// that are already dense 411 us), 17408 x 5120 204 us (237), 5120 x 5120 71 us (62); 77 rows of
// 4096 x 24576 42 us, 12288 x 4096 22 us.  The form with codes in registers took 540, 260, 105 and 87, 31 us for
// the same tiles.  What bounds it at many rows is shared (counters, the first of these shapes with the
// activation): matrix instructions 42 % of the SIMDs' cycles, other vector instructions 38 %, the LDS busy for 50 % - half of that
// bank conflicts - at 1.9 of 2.4 GHz (power); with no dequantisation at all the same loop is 20 % faster.
// At few rows it is latency - two memory round trips before the first product and one for the slices, a third of the
// waves' time - and the LDS: 77 rows of 4096 x 24576 matrix 24 %, vector 37 %, LDS 51 %.
// The activation's exponential is expf as in its other forms; 64 of them per lane behind the last stage cost 1 %.
#include "dflash_common.h"
#include "qmm_stream_device.h"

namespace dflash {
namespace rows {

constexpr int kWaves = 4;      // side by side
constexpr int kStageK = 64;    // k per stage and set of waves

struct Args {
  const uint16_t* x;
  const uint32_t* w;
  const uint16_t* scales;
  const uint16_t* biases;
  uint16_t* y;
  float* partials;      // [cut tile][slice][tile of 16x16 in the workgroup][thread][4]
  uint32_t* counters;   // one per cut tile, zero between calls
  int M, K, N;
  int group_shift;      // log2(group size)
  int tiles_m, tiles;
  int whole, slices;    // tiles computed in one piece; slices of K of the others
  int stages;           // ceil(K / (64 KG))
};

template <bool FP16>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (FP16) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{a, b}), f16x2_t));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{a, b}), bf16x2_t));
  }
}
template <bool FP16>
__device__ __forceinline__ float round16(float v) {
  if constexpr (FP16) return (float)(_Float16)v;
  else return (float)(__bf16)v;
}
__device__ __forceinline__ float code_fma(uint32_t pair, int hi, float s24, float b) {
  const f16x2_t h = __builtin_bit_cast(f16x2_t, pair);
  return __builtin_fmaf((float)h[hi], s24, b);
}
// eight codes of one word (k ascending from the low nibble) -> eight values of the activation type; s24 and s20
// are the scale times 2^24 and 2^20 (a code in bits 4 .. 7 of a half word is 16 times one in bits 0 .. 3)
template <bool FP16>
__device__ __forceinline__ uint4 dequant8(uint32_t w, float s24, float s20, float b, uint32_t mask0, uint32_t mask4) {
  const uint32_t w8 = w >> 8;
  const uint32_t p0 = w & mask0, p1 = w & mask4, p2 = w8 & mask0, p3 = w8 & mask4;  // (k0,k4) (k1,k5) ..
  uint4 r;
  r.x = pack2<FP16>(code_fma(p0, 0, s24, b), code_fma(p1, 0, s20, b));
  r.y = pack2<FP16>(code_fma(p2, 0, s24, b), code_fma(p3, 0, s20, b));
  r.z = pack2<FP16>(code_fma(p0, 1, s24, b), code_fma(p1, 1, s20, b));
  r.w = pack2<FP16>(code_fma(p2, 1, s24, b), code_fma(p3, 1, s20, b));
  return r;
}
template <bool FP16>
__device__ __forceinline__ float sb_value(uint32_t h) {
  return FP16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
}

// KG: sets of four waves, each with its 64 k of a stage.
// SILU_MUL: W holds the gate rows and, behind them, the up rows of an MLP, y[M, N / 2] is silu(gate) * up with every
// operator's rounding to the activation type.  Half of a wave's tiles are gate columns, the others the up
// columns of the same lanes.
template <bool FP16, bool SB_FP16, int MT, int NT, int KG, bool SILU_MUL>
__global__ __launch_bounds__(256 * KG, 2) void qmm_rows_kernel(Args a) {
  using A = stream::Act<FP16>;
  constexpr int kThreads = 256 * KG;
  constexpr int BM = 16 * MT, BN = kWaves * 16 * NT;
  constexpr int kXBytes = KG * BM * 128, kWBytes = KG * BN * 32;
  constexpr int kFrontBytes = 2 * kXBytes + 3 * kWBytes;
  constexpr int kSbBytes = 2 * BN * 16;  // scales and biases of eight groups
  constexpr int kXRows = kThreads / (8 * KG), XL = (BM + kXRows - 1) / kXRows;  // 16-byte pieces of x per thread
  constexpr int kWRows = kThreads / (2 * KG), WL = (BN + kWRows - 1) / kWRows;  // ... of codes
  constexpr int SL = (2 * BN + kThreads - 1) / kThreads;                        // ... of scales and biases
  extern __shared__ __attribute__((aligned(1024))) char lds[];  // x of 2 stages, codes of 3, 2 chunks of scales and biases
  __shared__ uint32_t s_last;
  char* const w_lds = lds + 2 * kXBytes;
  char* const sb_lds = lds + kFrontBytes;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
  const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
  const int li = lane & 15, kq = lane >> 4;
  // neighbours in tile order (same columns, other rows) behind one L2; the whole tiles are dispatched first
  const bool cut = (int)blockIdx.x >= a.whole;
  const int part = cut ? (int)gridDim.x - a.whole : a.whole, at = (int)blockIdx.x - (cut ? a.whole : 0);
  const int wg = part % 8 == 0 ? (at % 8) * (part / 8) + at / 8 : at;
  const int slices = cut ? a.slices : 1, slice = wg % slices, cut_tile = wg / slices;
  const int tile = cut ? a.whole + cut_tile : wg;
  const int st0 = a.stages * slice / slices, st1 = a.stages * (slice + 1) / slices;  // (at most 16 slices)
  const int nb = tile / a.tiles_m, mb = tile - nb * a.tiles_m;
  const int m0 = mb * BM, n0 = nb * BN;
  const int G = a.K >> a.group_shift;
  uint32_t mask0 = 0x000F000Fu, mask4 = 0x00F000F0u;
  asm volatile("" : "+s"(mask0), "+s"(mask4));

  constexpr int kTiles = SILU_MUL ? NT / 2 : NT;  // tiles of output columns per wave
  static_assert(!SILU_MUL || NT % 2 == 0, "gate and up tiles come in pairs");
  const int out_cols = SILU_MUL ? a.N / 2 : a.N;
  // Where row r of the workgroup's part of W sits in LDS: tile t of a wave holds rows 4 T (i / 4) + 4 t + i % 4 of its 16 T
  // (T = kTiles), i = 0 .. 15, one after the other.
  auto position = [](int r) __attribute__((always_inline)) {
    const int half = SILU_MUL ? r / (BN / 2) : 0;
    r -= half * (BN / 2);
    const int w = r / (16 * kTiles), c = r % (16 * kTiles);
    return w * (16 * NT) + (half * kTiles + (c >> 2) % kTiles) * 16 + (c / (4 * kTiles)) * 4 + (c & 3);
  };
  // ... and which row of W it is
  auto row_of_w = [&](int r) __attribute__((always_inline)) {
    const int half = SILU_MUL ? r / (BN / 2) : 0;
    int n = (SILU_MUL ? n0 / 2 : n0) + r - half * (BN / 2);
    n = n < out_cols ? n : out_cols - 1;
    return n + half * out_cols;
  };

  // this thread's pieces of a stage: uniform bases, 32-bit byte offsets from them
  const char* const xbase = (const char*)(a.x + (size_t)m0 * a.K);
  const char* const wbase = (const char*)a.w + (size_t)(SILU_MUL ? 0 : n0) * (a.K >> 1);
  const int xg = tid % (8 * KG), xr = tid / (8 * KG), wg16 = tid % (2 * KG), wr = tid / (2 * KG);
  uint32_t xo[XL];
  size_t wo[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    int row = xr + kXRows * i;
    row = m0 + row < a.M ? row : a.M - 1 - m0;
    xo[i] = (uint32_t)row * (uint32_t)a.K * 2u;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int row = row_of_w(wr + kWRows * i < BN ? wr + kWRows * i : BN - 1) - (SILU_MUL ? 0 : n0);
    wo[i] = (size_t)row * ((uint32_t)a.K >> 1);
  }
  static_assert(WL <= 2, "two pieces of codes per thread at most");
  uint4 xv[XL], wv0, wv1, sv[SL];
  auto load_x = [&](int st) __attribute__((always_inline)) {
    const int kx = st * (kStageK * KG) + 8 * xg;
    const uint32_t xk = kx < a.K ? 2u * kx : 0u;
#pragma unroll
    for (int i = 0; i < XL; ++i) xv[i] = *reinterpret_cast<const uint4*>(xbase + (xo[i] + xk));
    if (kx >= a.K) {  // k past the end of the rows: zeros on this side are enough
#pragma unroll
      for (int i = 0; i < XL; ++i) xv[i] = make_uint4(0u, 0u, 0u, 0u);
    }
  };
  auto load_w = [&](int st) __attribute__((always_inline)) {
    const int kw = st * (kStageK * KG) + 32 * wg16;
    const uint32_t wk = kw < a.K ? (uint32_t)kw >> 1 : 0u;
    wv0 = *reinterpret_cast<const uint4*>(wbase + (wo[0] + wk));
    if constexpr (WL == 2) wv1 = *reinterpret_cast<const uint4*>(wbase + (wo[WL - 1] + wk));
  };
  auto store_x = [&](int buf) __attribute__((always_inline)) {
    char* const xs = lds + buf * kXBytes + (xg >> 3) * (BM * 128);
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int row = xr + kXRows * i;
      if (BM % kXRows == 0 || row < BM) *reinterpret_cast<uint4*>(xs + row * 128 + (((xg & 7) ^ ((row >> 1) & 7)) << 4)) = xv[i];
    }
  };
  auto store_w = [&](int buf) __attribute__((always_inline)) {
    char* const ws = w_lds + buf * kWBytes + (wg16 >> 1) * (BN * 32) + (wg16 & 1) * 16;
    if (BN >= kWRows || wr < BN) *reinterpret_cast<uint4*>(ws + position(wr) * 32) = wv0;
    if constexpr (WL == 2) {
      if (BN % kWRows == 0 || wr + kWRows < BN) *reinterpret_cast<uint4*>(ws + position(wr + kWRows) * 32) = wv1;
    }
  };
  // a chunk is the scales and biases of eight groups (16 bytes) of every row
  auto load_chunk = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      const int e = tid + kThreads * i, r = e % BN;
      const int n = row_of_w(r);
      const uint16_t* src = (e < BN ? a.scales : a.biases) + (size_t)n * G;
      if (8 * chunk + 8 <= G) {
        struct __attribute__((packed, aligned(2))) Loose { uint32_t a, b, c, d; };  // (rows of scales start on any element)
        const Loose v = *reinterpret_cast<const Loose*>(src + 8 * chunk);
        sv[i] = make_uint4(v.a, v.b, v.c, v.d);
      } else {
        uint32_t h[8];
#pragma unroll
        for (int g = 0; g < 8; ++g) h[g] = src[8 * chunk + g < G ? 8 * chunk + g : G - 1];
        sv[i] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
      }
    }
  };
  auto store_chunk = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      const int e = tid + kThreads * i;
      if ((2 * BN) % kThreads == 0 || e < 2 * BN)
        *reinterpret_cast<uint4*>(sb_lds + buf * kSbBytes + (e < BN ? 0 : BN * 16) + position(e % BN) * 16) = sv[i];
    }
  };
  const int stages_per_chunk = (8 << a.group_shift) / (kStageK * KG);

  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  int chunk = st0 / stages_per_chunk;  // of the stage whose codes are read next, and its place in the chunk
  int in_chunk = st0 - chunk * stages_per_chunk;
  const int last_chunk = (a.stages - 1) / stages_per_chunk;
  int cbuf = 0, wbuf = 0;  // buffers of that stage
  // lane addresses inside a stage
  const char* const xrd = lds + kg * (BM * 128) + li * 128;
  const char* const wrd = w_lds + kg * (BN * 32) + (wave * (16 * NT) + li) * 32 + kq * 8;
  const char* const srd = sb_lds + (wave * (16 * NT) + li) * 16;
  uint2 wc[NT];
  float sc[NT], sc16[NT], bc[NT];
  auto read_codes = [&]() __attribute__((always_inline)) {
    // lane group kq multiplies k = 16 kq .. 16 kq + 15 of its 64: words 2 kq and 2 kq + 1 of a row
    const int g = ((in_chunk * KG + kg) * kStageK + 16 * kq) >> a.group_shift;
    const char* const sp = srd + cbuf * kSbBytes + g * 2;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      wc[t] = *reinterpret_cast<const uint2*>(wrd + wbuf * kWBytes + t * 512);
      const float scale = sb_value<SB_FP16>(*reinterpret_cast<const uint16_t*>(sp + t * 256));
      sc[t] = scale * 16777216.0f, sc16[t] = scale * 1048576.0f;
      bc[t] = sb_value<SB_FP16>(*reinterpret_cast<const uint16_t*>(sp + BN * 16 + t * 256));
    }
  };
  uint4 wf[2][NT];
  // Half a stage: the products with the weights in wf[j] and, spread over their matrix instructions, the
  // dequantisation of the other half.  x is read two rows of tiles ahead.
  constexpr int kAhead = NT == 4 ? 2 : 4;  // rows of tiles of x read ahead
  uint4 xf[kAhead + 1];
  auto first_x = [&](int j, int xbuf) __attribute__((always_inline)) -> const char* {
    const char* const xp = xrd + xbuf * kXBytes + (((2 * kq + j) ^ (li >> 1)) << 4);
#pragma unroll
    for (int i = 0; i < kAhead && i < MT; ++i) xf[i] = *reinterpret_cast<const uint4*>(xp + i * 2048);
    return xp;
  };
  auto half_stage = [&](int j, const char* xp) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (i + kAhead < MT) xf[(i + kAhead) % (kAhead + 1)] = *reinterpret_cast<const uint4*>(xp + (i + kAhead) * 2048);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[i][t] = A::mfma(wf[j][t], xf[i % (kAhead + 1)], acc[i][t]);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) wf[j ^ 1][t] = dequant8<FP16>(j == 0 ? wc[t].y : wc[t].x, sc[t], sc16[t], bc[t], mask0, mask4);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (i + kAhead < MT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, (20 + MT - 1) / MT, 0);
      }
    }
    // (used in the next stage only, the weights would be dequantised there)
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(wf[j ^ 1][t].x), "+v"(wf[j ^ 1][t].y), "+v"(wf[j ^ 1][t].z), "+v"(wf[j ^ 1][t].w));
    __builtin_amdgcn_sched_barrier(0);
  };

  load_chunk(chunk);
  load_w(st0);
  load_x(st0);
  store_chunk(0);
  store_w(0);
  load_w(st0 + 1);
  store_x(0);
  store_w(1);
  if (chunk < last_chunk) {
    load_chunk(chunk + 1);
    store_chunk(1);
  }
  load_x(st0 + 1);
  load_w(st0 + 2);
  __syncthreads();
  read_codes();
#pragma unroll
  for (int t = 0; t < NT; ++t) wf[0][t] = dequant8<FP16>(wc[t].x, sc[t], sc16[t], bc[t], mask0, mask4);
  for (int st = st0; st < st1; ++st) {
    const int xbuf = (st - st0) & 1;
    const bool brings_chunk = in_chunk == 0 && st != st0 && chunk < last_chunk;
    if (brings_chunk) load_chunk(chunk + 1);
    half_stage(0, first_x(0, xbuf));
    // What was asked for a stage ago goes to LDS in the middle of this one, and the next requests leave: a
    // whole stage for the latency of memory, and no wave waits at the barrier for another one's loads.
    // (Behind the last stage: loads of valid addresses, stores to buffers that nobody reads.)
    store_x(xbuf ^ 1);
    store_w(wbuf == 0 ? 2 : wbuf - 1);
    load_x(st + 2);
    load_w(st + 3);
    // the codes of the next stage (behind the last one: of some stage that is in LDS, not used)
    const int cbuf_now = cbuf;
    if (++wbuf == 3) wbuf = 0;
    if (++in_chunk == stages_per_chunk) {
      in_chunk = 0;
      ++chunk;
      cbuf ^= 1;
    }
    const char* const xp = first_x(1, xbuf);
    read_codes();
    half_stage(1, xp);
    if (brings_chunk) store_chunk(cbuf_now ^ 1);
    __syncthreads();
  }

  if constexpr (KG == 2) {
    // the second set hands its sums over through LDS, as many rows of tiles at a time as fit the stages
    constexpr int kPer = kFrontBytes / (4096 * NT) < MT ? kFrontBytes / (4096 * NT) : MT;
    f32x4_t* const red = reinterpret_cast<f32x4_t*>(lds);
    const int t256 = tid & 255;
#pragma unroll
    for (int i0 = 0; i0 < MT; i0 += kPer) {
      if (i0 > 0) __syncthreads();
      if (kg == 1) {
#pragma unroll
        for (int i = i0; i < i0 + kPer && i < MT; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t) red[((i - i0) * NT + t) * 256 + t256] = acc[i][t];
      }
      __syncthreads();
      if (kg == 0) {
#pragma unroll
        for (int i = i0; i < i0 + kPer && i < MT; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[i][t] += red[((i - i0) * NT + t) * 256 + t256];
      }
    }
  }

  // accumulator r of lane (li, kq), tile (i, t): row m0 + 16 i + li, column 16 T wave + 4 T kq + 4 t + r of the workgroup's
  auto emit = [&](int i, const f32x4_t (&v)[NT]) __attribute__((always_inline)) {
    const int m = m0 + 16 * i + li, n = (SILU_MUL ? n0 / 2 : n0) + wave * (16 * kTiles) + 4 * kTiles * kq;
    if (m >= a.M) return;
    uint16_t* dst = a.y + (size_t)m * out_cols + n;
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      f32x4_t o = v[t];
      if constexpr (SILU_MUL) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float g = round16<FP16>(v[t][r]), u = round16<FP16>(v[t + kTiles][r]);
          const float s = round16<FP16>(1.0f / (1.0f + expf(-g)));
          o[r] = round16<FP16>(g * s) * u;
        }
      }
      const uint2 w = make_uint2(pack2<FP16>(o[0], o[1]), pack2<FP16>(o[2], o[3]));
      if (n + 4 * t < out_cols) *reinterpret_cast<uint2*>(dst + 4 * t) = w;
    }
  };
  if (slices == 1) {
    if (kg == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i) emit(i, acc[i]);
    }
    return;
  }
  // Partial tiles are written through to and read from the level all XCDs share (sc1, as in the streaming kernel).
  constexpr size_t kTileFloats = (size_t)BM * BN;
  float* const first = a.partials + (size_t)cut_tile * slices * kTileFloats;
  if (kg == 0) {
    float* mine = first + slice * kTileFloats + (tid & 255) * 4;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) stream::store_partial(mine + (i * NT + t) * 1024, acc[i][t]);
  }
  // every wave's stores are acknowledged before the arrival is counted
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) s_last = atomicInc(&a.counters[cut_tile], (uint32_t)(slices - 1)) == (uint32_t)(slices - 1);
  __syncthreads();
  if (!s_last || kg != 0) return;
  // in order of k; a row of tiles of every slice is asked for before the first is looked at
  const auto parts = __builtin_amdgcn_make_buffer_rsrc(first, 0, 0x7FFFFFFF, 0x00027000);
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    f32x4_t sum[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) sum[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < slices; c0 += 4) {
      f32x4_t v[4][NT];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int cc = c0 + c < slices ? c0 + c : slices - 1;
#pragma unroll
        for (int t = 0; t < NT; ++t)
          v[c][t] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
              parts, (uint32_t)(tid * 16 + (i * NT + t) * 4096 + cc * (kTileFloats * 4)), 0, 16));
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c0 + c < slices) {
#pragma unroll
          for (int t = 0; t < NT; ++t) sum[t] += v[c][t];
        }
    }
    emit(i, sum);
  }
}

// The tile shapes there are: columns (16 NT a wave) for a height, and the one with a single set of waves for calls with
// many tiles.
template <bool FP16>
const void* kernel_for(int mt, int nt, int kg, bool mixed, bool silu_mul) {
#define DFLASH_ROWS_PICK(MT, NT, KG) \
  if (mt == MT && nt == NT && kg == KG && !mixed && !silu_mul) return (const void*)qmm_rows_kernel<FP16, FP16, MT, NT, KG, false>;
#define DFLASH_ROWS_PICK_SILU(MT, NT, KG) \
  if (mt == MT && nt == NT && kg == KG && !mixed && silu_mul) return (const void*)qmm_rows_kernel<FP16, FP16, MT, NT, KG, true>;
#define DFLASH_ROWS_PICK_MIXED(MT, NT, KG) \
  if (mt == MT && nt == NT && kg == KG && mixed && !silu_mul) return (const void*)qmm_rows_kernel<FP16, !FP16, MT, NT, KG, false>;
  DFLASH_ROWS_PICK(1, 1, 2)
  DFLASH_ROWS_PICK(2, 1, 2) DFLASH_ROWS_PICK(2, 2, 2) DFLASH_ROWS_PICK_SILU(2, 2, 2)
  DFLASH_ROWS_PICK(3, 1, 2) DFLASH_ROWS_PICK(3, 2, 2) DFLASH_ROWS_PICK_SILU(3, 2, 2)
  DFLASH_ROWS_PICK(4, 1, 2) DFLASH_ROWS_PICK(4, 2, 2) DFLASH_ROWS_PICK_SILU(4, 2, 2)
  DFLASH_ROWS_PICK(5, 1, 2) DFLASH_ROWS_PICK(5, 2, 2) DFLASH_ROWS_PICK_SILU(5, 2, 2)
  DFLASH_ROWS_PICK(6, 1, 2) DFLASH_ROWS_PICK(6, 2, 2) DFLASH_ROWS_PICK_SILU(6, 2, 2)
  DFLASH_ROWS_PICK(7, 1, 2) DFLASH_ROWS_PICK(7, 2, 2) DFLASH_ROWS_PICK_SILU(7, 2, 2)
  DFLASH_ROWS_PICK(8, 1, 2) DFLASH_ROWS_PICK(8, 2, 2) DFLASH_ROWS_PICK_SILU(8, 2, 2)
  DFLASH_ROWS_PICK(8, 3, 2) DFLASH_ROWS_PICK(8, 4, 2) DFLASH_ROWS_PICK_SILU(8, 4, 2)
  DFLASH_ROWS_PICK(8, 3, 1) DFLASH_ROWS_PICK(8, 4, 1) DFLASH_ROWS_PICK_SILU(8, 4, 1)
  // scales of the other 16-bit type: a few shapes
  DFLASH_ROWS_PICK_MIXED(2, 1, 2) DFLASH_ROWS_PICK_MIXED(4, 2, 2) DFLASH_ROWS_PICK_MIXED(8, 2, 2)
#undef DFLASH_ROWS_PICK
#undef DFLASH_ROWS_PICK_SILU
#undef DFLASH_ROWS_PICK_MIXED
  return nullptr;
}
constexpr int lds_bytes(int mt, int nt, int kg) { return kg * (2 * 16 * mt * 128 + 3 * 64 * nt * 32) + 2 * 2 * 64 * nt * 16; }

struct Plan {
  int mt, nt, kg, whole, slices, tiles_m, tiles, stages, grid;
  size_t workspace;
};

constexpr size_t kCounterBytes = 64 * 1024;

bool covers(int M, int K, int N, int group_size, bool mixed, int epilogue) {
  if (epilogue != DFLASH_QMM_EPILOGUE_NONE && (epilogue != DFLASH_QMM_EPILOGUE_SILU_MUL || mixed || N % 32 != 0)) return false;
  return M > 0 && K > 0 && N > 0 && (group_size == 32 || group_size == 64 || group_size == 128) && K % group_size == 0 &&
         N % 16 == 0;
}

// Which tile, how many slices of K: the least of a model of the time, fitted to 2757 measured combinations (8 shapes of
// 1 to 178 M weights, 20 to 1024 rows; 8 % rms, and what it picks is within 1 % of the best measured one on
// average, 12 % at worst).  A stage of 64 KG columns of K costs a fixed part (barrier, latency) and parts that go with
// the columns (codes to dequantise), the rows (x) and their product (matrix work); a workgroup with two sets of waves
// has a CU to itself, those with one share it in pairs.
// The last round of more tiles than fit at once is cut with the tile left as it is: matrix work that fills the chip
// runs against its power, so a smaller tile that fills it better gains nothing (5120 x 12352 over 1024 rows: 65 x 8
// tiles of 192 columns, 8 of them cut, 190 us; 49 x 8 of 256, uncut, 179).  Partial tiles behind whole rounds meet the
// memory busy, 3 TB/s for their way out and back: of 5120 x 34816, 64 of 1088 in four slices save 24 us, of
// 5120 x 12352, 136 of 392 in three slices nothing.
Plan make_plan(int M, int K, int N, int cus, bool mixed, bool silu_mul) {
  auto microseconds = [cus](const Plan& p) {
    const int slots = cus * (p.kg == 1 ? 2 : 1);
    const double stage = 0.134 + 0.1256 * p.nt + 0.0463 * p.mt + 0.0342 * p.mt * p.nt;
    const int whole = p.slices > 1 ? p.whole / slots : p.tiles / slots;  // rounds
    const int parts = p.grid - whole * slots, full = parts / slots, rest = parts - full * slots;
    // a last round with one workgroup per CU where there is room for two is the faster one
    const double rounds = full + (rest == 0 ? 0. : p.kg == 1 && rest <= cus ? 0.62 : 1.);
    double us = 7.55 + whole * (p.stages * stage - 2.89) + rounds * ((p.stages + p.slices - 1) / p.slices * stage - 2.89);
    if (p.slices > 1) us += 1.48 + 0.113 * p.slices * p.mt * p.nt;
    if (p.slices > 1 && whole > 0) us += parts * (16. * p.mt * 64 * p.nt * 8) / 3e6;
    return us;
  };
  Plan best{};
  double best_us = 0.;
  for (int mt = 1; mt <= 8; ++mt) {
    for (int nt = 1; nt <= 4; ++nt) {
      for (int kg = 1; kg <= 2; ++kg) {
        if (kernel_for<false>(mt, nt, kg, mixed, silu_mul) == nullptr) continue;
        Plan p{};
        p.mt = mt, p.nt = nt, p.kg = kg;
        p.tiles_m = (M + 16 * mt - 1) / (16 * mt);
        p.tiles = p.tiles_m * ((N + 64 * nt - 1) / (64 * nt));
        p.stages = (K + kStageK * kg - 1) / (kStageK * kg);
        const int slots = cus * (kg == 1 ? 2 : 1);
        for (p.slices = 1; p.slices <= 16 && p.slices <= p.stages; ++p.slices) {
          if (p.slices > 1 && (p.tiles * p.slices > slots || p.tiles > (int)(kCounterBytes / 4))) break;
          p.whole = p.slices > 1 ? 0 : p.tiles;
          p.grid = p.tiles * p.slices;
          const double us = microseconds(p);
          if (best.grid == 0 || us < best_us) best = p, best_us = us;
        }
      }
    }
  }
  const int slots = cus * (best.kg == 1 ? 2 : 1), cut = best.tiles % slots;
  if (best.slices == 1 && best.tiles > slots && cut > 0) {
    Plan p = best;
    p.whole = best.tiles - cut;
    for (p.slices = 2; p.slices <= 16 && p.slices <= p.stages && cut * p.slices <= 2 * slots; ++p.slices) {
      p.grid = p.whole + cut * p.slices;
      const double us = microseconds(p);
      if (us < best_us) best = p, best_us = us;
    }
  }
  best.workspace = best.slices > 1 ? kCounterBytes + (size_t)(best.grid - best.whole) * (16 * best.mt) * (64 * best.nt) * sizeof(float) : 0;
  return best;
}

// The last few plans of this thread: a model asks for the same ones over and over.
const Plan& plan(int M, int K, int N, int cus, bool mixed, bool silu_mul) {
  struct Entry {
    int M, K, N, cus, flags;
    Plan p;
  };
  static thread_local Entry cache[64] = {};
  const int flags = (mixed ? 2 : 0) | (silu_mul ? 1 : 0);
  Entry& e = cache[((unsigned)M * 2654435761u + (unsigned)K * 40503u + (unsigned)N * 69069u + (unsigned)flags) >> 26];
  if (e.M != M || e.K != K || e.N != N || e.cus != cus || e.flags != flags)
    e = Entry{M, K, N, cus, flags, make_plan(M, K, N, cus, mixed, silu_mul)};
  return e.p;
}

}  // namespace rows

int qmm_stream_grid();
}  // namespace dflash

extern "C" size_t dflash_qmm_rows_workspace_bytes(int M, int K, int N, int group_size, int act_dtype, int sb_dtype, int epilogue) {
  using namespace dflash;
  if (!rows::covers(M, K, N, group_size, act_dtype != sb_dtype, epilogue)) return 0;
  return rows::plan(M, K, N, qmm_stream_grid(), act_dtype != sb_dtype, epilogue != DFLASH_QMM_EPILOGUE_NONE).workspace;
}

extern "C" int dflash_qmm_rows(const void* x, const uint32_t* w_q, const void* scales, const void* biases, void* y,
                               void* workspace, size_t workspace_bytes, int M, int K, int N, int group_size,
                               int act_dtype, int sb_dtype, int epilogue, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(x && w_q && scales && biases && y, DFLASH_ERR_ARG, "dflash_qmm_rows: null operand");
  DFLASH_REQUIRE((act_dtype == DFLASH_BF16 || act_dtype == DFLASH_FP16) && (sb_dtype == DFLASH_BF16 || sb_dtype == DFLASH_FP16),
                 DFLASH_ERR_ARG, "dflash_qmm_rows: activations and scales must be bf16/fp16");
  const bool mixed = act_dtype != sb_dtype, silu_mul = epilogue != DFLASH_QMM_EPILOGUE_NONE;
  DFLASH_REQUIRE(rows::covers(M, K, N, group_size, mixed, epilogue), DFLASH_ERR_SHAPE,
                 "dflash_qmm_rows: need M > 0, group_size in {32,64,128}, K %% group_size == 0, N %% 16 == 0 (32 and one dtype "
                 "with the silu-mul epilogue) (M=%d K=%d N=%d gs=%d)", M, K, N, group_size);
  DFLASH_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)w_q % 16) == 0 && ((uintptr_t)y % 8) == 0, DFLASH_ERR_ARG,
                 "dflash_qmm_rows: x and w_q must be 16-byte aligned");
  const rows::Plan& p = rows::plan(M, K, N, qmm_stream_grid(), mixed, silu_mul);
  DFLASH_REQUIRE(p.workspace == 0 || (workspace && workspace_bytes >= p.workspace), DFLASH_ERR_WORKSPACE,
                 "dflash_qmm_rows: workspace of %zu bytes needed, %zu given", p.workspace, workspace ? workspace_bytes : (size_t)0);
  rows::Args a;
  a.x = (const uint16_t*)x; a.w = w_q; a.scales = (const uint16_t*)scales; a.biases = (const uint16_t*)biases;
  a.y = (uint16_t*)y;
  a.counters = (uint32_t*)workspace;
  a.partials = workspace ? (float*)((char*)workspace + rows::kCounterBytes) : nullptr;
  a.M = M; a.K = K; a.N = N;
  a.group_shift = group_size == 32 ? 5 : group_size == 64 ? 6 : 7;
  a.tiles_m = p.tiles_m; a.tiles = p.tiles; a.whole = p.whole; a.slices = p.slices; a.stages = p.stages;
  const bool fp16 = act_dtype == DFLASH_FP16;
  const void* fn = fp16 ? rows::kernel_for<true>(p.mt, p.nt, p.kg, mixed, silu_mul)
                        : rows::kernel_for<false>(p.mt, p.nt, p.kg, mixed, silu_mul);
  const int lds_bytes = rows::lds_bytes(p.mt, p.nt, p.kg);
  static bool attr_set[kMaxDevices][8][9][5][3] = {};
  const int dev = current_device_slot();
  if (lds_bytes > 48 * 1024) {
    bool& set = attr_set[dev][4 * silu_mul + 2 * fp16 + mixed][p.mt][p.nt][p.kg];
    if (!set || dev == kMaxDevices - 1) {
      DFLASH_HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes));
      set = true;
    }
  }
  void* args[] = {&a};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)p.grid), dim3(256 * p.kg), args, (size_t)lds_bytes, (hipStream_t)stream));
  return DFLASH_OK;
}
