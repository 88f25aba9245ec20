// 4-bit affine matmul for any number of rows, y[M,N] = x[M,K] . round(s*q + b)^T (gfx950): prompts,
// and every other call the 16-row kernels do not serve.
//
// What the reference leaves to mx.quantized_matmul (dflash_mlx/verify_qmm.py:277-280).  A weight is
// dequantised to the activation type as the array-op form of this package does it (s*q + b in
// fp32, rounded once) and multiplied on the matrix cores with fp32 accumulation.
//
//  * A wave owns whole columns: W waves side by side, each 32*NT columns wide and all 32*MT rows high, so that a
//    weight is dequantised once per 32*MT rows.  KG sets of such waves take 64 k of every stage each and add
//    their sums up through LDS at the end: eight waves on a CU without cutting the result any smaller.
//  * Matrix instructions of 32 x 32 x 16.  One takes the issue port of its SIMD for 8 cycles and the matrix pipe for
//    32 (16 x 16 x 32: 8 and 16, for half the work), and a vector instruction takes the port for 4: six of them hide beside a large
//    one, two beside a small one (measured: 33.9 and 42.7 cycles with 6 and 8 beside a large one; 17.4, 21.8 and 25.7 with 2, 3 and 4
//    beside a small one).  Dequantisation is 5 to 6 for MT = 4.  The order of instructions is spelled out per step
//    of 16 k: a few vector instructions behind each matrix instruction.
//  * x and codes go from memory to LDS past the registers: a write of 16 bytes per lane takes the LDS 14 cycles, a read 4,
//    and the form of this kernel that loaded to registers spent an eighth of its time on the writes.  Lane i of a request lands
//    at 16 i, so the places that keep reads free of bank conflicts are made by what each lane asks for.  A read of 16
//    bytes per lane serves lanes {0-3, 12-15, 20-23, 24-27} together, then {4-7, 8-11, 16-19, 28-31} and so on.
//  * dequantisation: code q sits in the low bits of a half word; as an fp16 subnormal that half is
//    q 2^-24, so fma_mix(half, s 2^24, b) is s q + b in one instruction and exact up to its one
//    rounding; the conversion to the activation type packs two at a time: 19 vector instructions per
//    8 weights.
//  * W is the A operand (rows of the tile = columns of y), x the B operand, and the columns of a
//    tile are dealt so that a lane ends up with 16 consecutive columns of one row.
//  * Where the tiles do not fill the chip, K is cut into slices: workgroups leave fp32 partial tiles in
//    the workspace, and whoever arrives last at a tile adds them in order of k.  Nobody waits.  Deterministic.
//    Of more tiles than the chip takes at once, only those of the last, incomplete round are cut.
//
// Measured (us, group 64; before: 16 x 16 x 32 instructions, loads to registers): 1024 rows of 5120 x 34816 with the
// activation 398 -> 335 (1.09 PFLOP/s), 17408 x 5120 207 -> 184, 5120 x 12352 164 -> 134; 200 rows of 4096 x 4096 22.6 -> 17.5; 77 rows
// of 4096 x 24576 with the activation 35.7 -> 29.0, 12288 x 4096 24.9 -> 20.9; 20 rows of 5120 x 12352 21.4 -> 18.3, of 1024 x 1024 5.9 -> 5.7.
// Slower than that form: 77 to 128 rows of 3072 x 1024, 6 to 9 % when that was measured.  (17 to 48 rows of nearly every matrix are now the kernel's with
// weights in registers, qmm_resident.hip.)
// With the waves meeting before a stage's last step, and scales that go past the registers, before / after: 400 rows of 4096 x 2304 19.5 -> 16.9, 600
// of 3072 x 9216 48.4 -> 45.6, 77 of 12288 x 4096 23.5 -> 22.4, 1024 of 5120 x 12352 136.4 -> 132.8; 16 calls of 20 to 1024 rows 2 %.
// What bounds it at many rows: the matrix pipes are busy for 60 to 67 % of the cycles at 2.0 to 2.1 of 2.4 GHz (power); with no requests
// to memory at all the loop that met behind a stage's last step was 15 to 20 % faster, with no dequantisation on top 2 to 10 %.  At few rows, by stamps
// in that loop: 3300 cycles of setup, requests and their latency before the first product, 5000 and more for the slices, and between them the issue port: two
// waves of (3,2,2,4) on a SIMD held it for 1930 of a stage's 3100 cycles (v_fma_mix and conversions take it for 4.3 cycles, v_fma_f32 and shifts for 2.4), a
// wave that is alone there issues every 5 cycles.  Turns at priority between the two changed nothing.  Counters of the loop as it is, 77 rows of
// 4096 x 24576 with the activation / of 12288 x 4096: vector 47 / 34 % of the time that the SIMDs hold waves, matrix 39 / 23, waves wait 32 / 44.
#include "glue_device.h"

#include "qmm_stream_device.h"
#include <algorithm>

namespace dflash {
int qmm_stream_grid();
// qmm_resident.hip: up to 80 rows
bool qmm_resident_rows_plan(int M, int K, int N, int group_size, bool silu_mul, int* chunks, int* slices, double* us, size_t* workspace);
int qmm_resident_rows_launch(const void* x, const void* w, const void* scales, const void* biases, void* y, void* workspace, int M, int K,
                             int N, int group_size, int dtype, bool silu_mul, int chunks, int slices, hipStream_t stream);

namespace rows {

constexpr int kStageK = 64;  // k per stage and set of waves

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
  int loose;            // scales and biases go to LDS by way of registers
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
// Codes 2 p and 2 p + 1 of one word (k ascending from the low nibble) -> two values of the activation type; s24 and s20
// are the scale times 2^24 and 2^20 (a code in bits 4 .. 7 of a half word is 16 times one in bits 0 .. 3)
template <bool FP16>
__device__ __forceinline__ uint32_t dequant2(uint32_t w, int p, float s24, float s20, float b, uint32_t mask0, uint32_t mask4) {
  const uint32_t v = p & 1 ? w >> 8 : w;  // halves (k0, k4), (k1, k5) or (k2, k6), (k3, k7)
  return pack2<FP16>(code_fma(v & mask0, p >> 1, s24, b), code_fma(v & mask4, p >> 1, s20, b));
}
template <bool FP16>
__device__ __forceinline__ uint4 dequant8(uint32_t w, float s24, float s20, float b, uint32_t mask0, uint32_t mask4) {
  return make_uint4(dequant2<FP16>(w, 0, s24, s20, b, mask0, mask4), dequant2<FP16>(w, 1, s24, s20, b, mask0, mask4),
                    dequant2<FP16>(w, 2, s24, s20, b, mask0, mask4), dequant2<FP16>(w, 3, s24, s20, b, mask0, mask4));
}
template <bool FP16>
__device__ __forceinline__ float sb_value(uint32_t h) {
  return FP16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
}

typedef __attribute__((ext_vector_type(16))) float f32x16_t;

template <bool FP16>
__device__ __forceinline__ f32x16_t mfma32(uint4 w, uint4 x, f32x16_t c) {
  if constexpr (FP16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, w), __builtin_bit_cast(f16x8_t, x), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), c, 0, 0, 0);
  }
}

// Lane i of the wave: 16 bytes from rsrc + voff + soff to LDS at lds + 16 i, past the registers.  The compiler counts neither the
// request nor what it writes: whoever reads that place waits with stage_done() first, and whoever asks for it to be filled again
// has met every wave that read it since (stage_done() or all_read(), whose clobber keeps reads on their side).  Requests and
// these two stay in the order they are written in, all being volatile.
__device__ __forceinline__ void request16(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n s_nop 0\n buffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "m0");
}
// All but the last LEFT requests of this wave have landed, its writes to LDS are done, and so have and are every other wave's.
template <int LEFT>
__device__ __forceinline__ void stage_done() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n s_barrier" ::"n"(LEFT) : "memory");
}

// What this wave has read from LDS is in registers, and so is what every other wave has.
__device__ __forceinline__ void all_read() { asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory"); }

template <int MT, int NT, int W, int KG>
struct Tile {
  static constexpr int kThreads = 64 * W * KG, BM = 32 * MT, BN = 32 * NT * W;
  static constexpr int kGroups = KG < 4 ? 8 : 4 * KG;  // whose scales and biases are brought at a time: two stages at least
  static constexpr int kXBytes = KG * BM * 128, kWBytes = KG * BN * 32, kSbBytes = 4 * BN * kGroups;
  static constexpr int kXBufs = 2, kWBufs = 3;  // (a third buffer of x changes nothing: 17408 x 5120 over 1024 rows 201 and 203 us)
  static constexpr int kFrontBytes = kXBufs * kXBytes + kWBufs * kWBytes;
  static constexpr int kLdsBytes = kFrontBytes + 2 * kSbBytes;
};

// KG: sets of W waves, each with its 64 k of a stage.
// SILU_MUL: W holds the gate rows and, behind them, the up rows of an MLP, y[M, N / 2] is silu(gate) * up with every
// operator's rounding to the activation type.  A wave's first tile is gate columns, its second the up columns of the same lanes.
template <bool FP16, bool SB_FP16, int MT, int NT, int W, int KG, bool SILU_MUL>
__global__ __launch_bounds__(64 * W * KG, 2) void qmm_rows_kernel(Args a) {
  using T = Tile<MT, NT, W, KG>;
  constexpr int BM = T::BM, BN = T::BN, kThreads = T::kThreads, kSet = 64 * W, kGroups = T::kGroups;
  constexpr int XB = T::kXBufs, WB = T::kWBufs;
  constexpr int kXReq = BM / (8 * W), kWReq = NT;  // requests of a wave for a stage: 8 rows of x, 64 / (2 KG) rows of codes each
  static_assert(BM % (8 * W) == 0 && (!SILU_MUL || NT == 2), "whole requests; gate and up tiles come in pairs");
  extern __shared__ __attribute__((aligned(1024))) char lds[];  // x [buffer][set][row] 128 bytes, codes [buffer][row] 32 KG bytes, scales and biases [2]
  char* const w_lds = lds + XB * T::kXBytes;
  char* const sb_lds = lds + T::kFrontBytes;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(stream::lds_address(lds));

  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, kq = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wid % W, kg = wid / W;
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
  const int out_cols = SILU_MUL ? a.N / 2 : a.N;
  // Row of W at place p of the workgroup's (tile p / 32, row i = p % 32 of it): accumulator r of lane (lr, kq) is row
  // i = 8 (r / 4) + 4 kq + r % 4, which stands for column 16 kq + r of the tile, so that a lane has 16 consecutive ones.
  auto first_row = [&](int t) __attribute__((always_inline)) {  // of tile t
    return SILU_MUL ? n0 / 2 + (t >> 1) * 32 + (t & 1) * out_cols : n0 + t * 32;
  };
  auto row_in_tile = [](int i) __attribute__((always_inline)) { return 16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3); };

  // ---- what this wave requests: x by descriptors of the workgroup's rows, codes of one tile at a time ---------------------
  const int rows_here = a.M - m0 < BM ? a.M - m0 : BM;
  const auto x_buf = __builtin_amdgcn_make_buffer_rsrc((void*)(a.x + (size_t)m0 * a.K), 0, (int)((uint32_t)rows_here * (uint32_t)a.K * 2u), 0x00027000);
  // x: request j brings rows 8 (kXReq wave + j) .. + 7 of this wave's set, piece c of a row to place c ^ (row / 2 % 8)
  uint32_t xo[kXReq];
#pragma unroll
  for (int j = 0; j < kXReq; ++j) {
    const int row = 8 * (kXReq * wave + j) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
    xo[j] = (uint32_t)(row < rows_here ? row : rows_here - 1) * (uint32_t)a.K * 2u + 128u * kg + 16u * c;
  }
  const uint32_t x_to = lds0 + kg * (BM * 128) + 1024 * kXReq * wave;
  const int tail = a.K % (kStageK * KG) != 0 ? a.stages - 1 : -1;
  // codes: a row has 2 KG pieces (32 k each); request j brings 32 / KG rows, piece u of row p to place u ^ f(p)
  constexpr int kPieces = 2 * KG, kWRows = 64 / kPieces;
  auto code_place = [](int p) __attribute__((always_inline)) { return KG == 8 ? p & 15 : KG == 4 ? (p >> 1) & 7 : KG == 2 ? (p >> 2) & 3 : (p >> 3) & 1; };
  uint32_t wo[kWReq];
  __amdgpu_buffer_rsrc_t w_buf[kWReq];
#pragma unroll
  for (int j = 0; j < kWReq; ++j) {
    const int p0 = kWRows * (kWReq * wid + j), p = p0 + lane / kPieces, u = (lane % kPieces) ^ code_place(p);
    const int first = __builtin_amdgcn_readfirstlane(first_row(p0 >> 5));
    int here = (SILU_MUL && first >= out_cols ? a.N : out_cols) - first;  // rows there are
    const bool none = here <= 0;
    here = here > 32 ? 32 : here;
    const int row = row_in_tile(p & 31);
    wo[j] = (uint32_t)(row < here ? row : none ? 0 : here - 1) * ((uint32_t)a.K >> 1) + 16u * u;
    const int from = none ? 0 : first;
    w_buf[j] = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)a.w + (size_t)from * (a.K >> 1)), 0,
                                                 (int)((uint32_t)(none ? 1 : here) * ((uint32_t)a.K >> 1)), 0x00027000);
  }
  const uint32_t w_to = lds0 + XB * T::kXBytes + 1024 * kWReq * wid;
  // Stages behind the last one are the last one again; k past the end of the rows reads zeros (an offset behind all of them).
  auto request_x = [&](int st, int buf, int j) __attribute__((always_inline)) {
    st = st < a.stages ? st : a.stages - 1;
    const int row = 8 * (kXReq * wave + j) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
    const bool past = st == tail && (st * KG + kg) * kStageK + 8 * c >= a.K;
    request16(x_buf, x_to + buf * T::kXBytes + 1024 * j, past ? 0x80000000u : xo[j], st * (2 * kStageK * KG));
  };
  auto request_w = [&](int st, int buf, int j) __attribute__((always_inline)) {
    st = st < a.stages ? st : a.stages - 1;
    const int p = kWRows * (kWReq * wid + j) + lane / kPieces, u = (lane % kPieces) ^ code_place(p);
    const bool past = st == tail && st * (kStageK * KG) + 32 * u >= a.K;
    request16(w_buf[j], w_to + buf * T::kWBytes + 1024 * j, past ? 0x80000000u : wo[j], st * (kStageK * KG / 2));
  };
  // a chunk is the scales and biases of kGroups groups of every row, 16 bytes for eight of them
  constexpr int kSbPieces = kGroups / 4 * BN, SL = (kSbPieces + kThreads - 1) / kThreads;
  static_assert(kSbPieces % 64 == 0, "whole waves of pieces");
  auto has_piece = [&](int i) __attribute__((always_inline)) { return kSbPieces % kThreads == 0 || 64 * wid + kThreads * i < kSbPieces; };
  uint4 sv[SL];
  auto load_chunk = [&](int chunk, uint4 (&sv)[SL]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      if (!has_piece(i)) break;  // (no load that its wave never looks at: the compiler waits for those where it next writes their registers.  33
                                  // rows of 3168 x 4112 in groups of 32 14.6 -> 13.6 us, 100 of 11904 x 2048 in groups of 128 20.5 -> 19.6)
      const int e = tid + kThreads * i, p = e % BN, g0 = kGroups * chunk + (e / (2 * BN)) * 8;
      int n = first_row(p >> 5) + row_in_tile(p & 31);
      const int end = SILU_MUL && ((p >> 5) & 1) ? a.N : out_cols;
      n = n < end ? n : end - 1;
      const uint16_t* src = ((e / BN) % 2 == 0 ? a.scales : a.biases) + (size_t)n * G;
      if (g0 + 8 <= G) {
        struct __attribute__((packed, aligned(2))) Loose { uint32_t a, b, c, d; };  // (rows of scales start on any element)
        const Loose v = *reinterpret_cast<const Loose*>(src + g0);
        sv[i] = make_uint4(v.a, v.b, v.c, v.d);
      } else {
        uint32_t h[8];
#pragma unroll
        for (int g = 0; g < 8; ++g) h[g] = src[g0 + g < G ? g0 + g : G - 1];
        sv[i] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
      }
    }
  };
  auto store_chunk = [&](int buf, const uint4 (&sv)[SL]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < SL; ++i)
      if (has_piece(i)) *reinterpret_cast<uint4*>(sb_lds + buf * T::kSbBytes + (tid + kThreads * i) * 16) = sv[i];
  };
  // The same past the registers, a request for 64 rows at a time: scales in registers made the compiler wait for every request in flight, codes
  // of the next stages included.  What is asked for behind the end of a row is never read (a.loose: where it would be, and where rows start
  // on odd elements).
  constexpr bool kDirect = BN % 64 == 0;
  const auto s_buf = __builtin_amdgcn_make_buffer_rsrc((void*)a.scales, 0, (int)((uint32_t)a.N * (uint32_t)G * 2u), 0x00027000);
  const auto b_buf = __builtin_amdgcn_make_buffer_rsrc((void*)a.biases, 0, (int)((uint32_t)a.N * (uint32_t)G * 2u), 0x00027000);
  const uint32_t sb_to = lds0 + T::kFrontBytes;
  auto request_chunk = [&](int chunk, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < (kSbPieces / 64 + W * KG - 1) / (W * KG); ++i) {
      const int r = wid + W * KG * i;
      if ((kSbPieces / 64) % (W * KG) != 0 && r >= kSbPieces / 64) break;
      const int p = 64 * r % BN + lane;
      int n = first_row(p >> 5) + row_in_tile(p & 31);
      const int end = SILU_MUL && ((p >> 5) & 1) ? a.N : out_cols;
      n = n < end ? n : end - 1;
      const uint32_t from = ((uint32_t)n * (uint32_t)G + (uint32_t)(kGroups * chunk + (64 * r / (2 * BN)) * 8)) * 2u;
      request16((64 * r / BN) % 2 == 0 ? s_buf : b_buf, sb_to + buf * T::kSbBytes + 1024 * r, from, 0);
    }
  };
  const bool loose = !kDirect || a.loose != 0;
  const int stages_per_chunk = (kGroups << a.group_shift) / (kStageK * KG);

  f32x16_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][t][r] = 0.f;

  int chunk = st0 / stages_per_chunk;  // of the stage whose codes are read next, and its place in the chunk
  int in_chunk = st0 - chunk * stages_per_chunk;
  const int last_chunk = (a.stages - 1) / stages_per_chunk;
  int cbuf = 0, wbuf = 0;  // buffers of that stage
  // Lane (lr, kq) multiplies k = 32 kq .. 32 kq + 31 of its set's 64: step s of a stage 32 kq + 8 s .. + 7.
  const char* xrd[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) xrd[s] = lds + kg * (BM * 128) + lr * 128 + (((4 * kq + s) ^ ((lr >> 1) & 7)) << 4);
  const char* const wrd = w_lds + (wave * (32 * NT) + lr) * (32 * KG) + (((2 * kg + kq) ^ code_place(lr)) << 4);
  const char* const srd = sb_lds + (wave * (32 * NT) + lr) * 16;
  uint4 wc[NT];
  uint32_t sraw[NT], braw[NT];
  float sc[NT], sc16[NT], bc[NT];
  auto read_codes = [&]() __attribute__((always_inline)) {
    const int g = ((in_chunk * KG + kg) * kStageK + 32 * kq) >> a.group_shift;
    const char* const sp = srd + cbuf * T::kSbBytes + (kGroups == 8 ? 0 : (g >> 3) * (32 * BN)) + (kGroups == 8 ? g : g & 7) * 2;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      wc[t] = *reinterpret_cast<const uint4*>(wrd + wbuf * T::kWBytes + t * (1024 * KG));
      sraw[t] = *reinterpret_cast<const uint16_t*>(sp + t * 512);
      braw[t] = *reinterpret_cast<const uint16_t*>(sp + BN * 16 + t * 512);
    }
  };
  auto take_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float scale = sb_value<SB_FP16>(sraw[t]);
      sc[t] = scale * 16777216.0f, sc16[t] = scale * 1048576.0f;
      bc[t] = sb_value<SB_FP16>(braw[t]);
    }
  };
  constexpr int kAhead = MT == 1 ? 3 : 1;  // steps that x is read ahead: a step of few products is shorter than the way to LDS
  uint4 wf[2][NT], xf[kAhead + 1][MT];
  auto read_x = [&](int s, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; ++i) xf[s & kAhead][i] = *reinterpret_cast<const uint4*>(xrd[s] + buf * T::kXBytes + i * 4096);
  };

  // ---- prologue ------------------------------------------------------------------------------------------------------------
#pragma unroll
  for (int j = 0; j < kWReq; ++j) request_w(st0, 0, j);
#pragma unroll
  for (int j = 0; j < kXReq; ++j) request_x(st0, 0, j);
#pragma unroll
  for (int j = 0; j < kWReq; ++j) request_w(st0 + 1, 1, j);
  const bool two_chunks = (chunk + 1) * stages_per_chunk < st1;
  if (loose) {
    uint4 sv_next[SL];
    load_chunk(chunk, sv);
    if (two_chunks) load_chunk(chunk + 1, sv_next);
    store_chunk(0, sv);
    if (two_chunks) store_chunk(1, sv_next);
  } else if constexpr (kDirect) {
    request_chunk(chunk, 0);
    if (two_chunks) request_chunk(chunk + 1, 1);
  }
  // (behind the scales in either form: the wait for those in registers is one for everything that was asked for before them)
#pragma unroll
  for (int j = 0; j < kWReq; ++j) request_w(st0 + 2, 2, j);
#pragma unroll
  for (int j = 0; j < kXReq; ++j) request_x(st0 + 1, 1, j);
  static_assert(WB == 3 && XB == 2, "the stages that are asked for ahead");
  stage_done<kWReq + kXReq>();
  read_codes();
#pragma unroll
  for (int s = 0; s < kAhead; ++s) read_x(s, 0);
  // The first stage asks for codes into the buffer that was just read, before its own meeting: the codes of a row of 2 KG pieces come
  // by requests of other waves than those that read them.  Without this meeting a wave that was held up between the two
  // multiplied with codes of stage st0 + 3 (seen while the requests stood before scales in registers, for whose registers the compiler
  // put a wait for all of memory right there: 9 of 64 calls differed from run to run).  It takes 0.1 us (100 rows of 512 x 2048 5.3 -> 5.4,
  // 150 of 2048 x 8192 14.1 -> 14.3, 200 of 4096 x 4096 18.6 -> 19.1, long calls as before).
  if constexpr (KG > 1) all_read();
  take_scales();
#pragma unroll
  for (int t = 0; t < NT; ++t) wf[0][t] = dequant8<FP16>(wc[t].x, sc[t], sc16[t], bc[t], mask0, mask4);

  int xbuf = 0;
  for (int st = st0; st < st1; ++st) {
    const bool brings_chunk = in_chunk == 0 && st != st0 && chunk < last_chunk;
    const int next_chunk = chunk + 1;
    if (brings_chunk && loose) load_chunk(next_chunk, sv);
    const int cbuf_now = cbuf, wbuf_now = wbuf;
    if (++wbuf == WB) wbuf = 0;
    if (++in_chunk == stages_per_chunk) {
      in_chunk = 0;
      ++chunk;
      cbuf ^= 1;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      // The next step's x; requests for later stages; the next stage's codes, whose first word the last step dequantises.  The waves meet before
      // the last step and not behind it: its operands are in registers, its products run while the next stage's first x is read, and the x of
      // the stage after that, whose place is free, has a whole stage to come.
      if (s == 3) {
        if (brings_chunk && loose) store_chunk(cbuf_now ^ 1, sv);
        // (the codes asked for in this stage may take another one; loads of scales among the requests make the wait longer, never shorter)
        stage_done<kWReq>();
#pragma unroll
        for (int q = 0; q < kAhead; ++q) read_x(q, xbuf ^ 1);
#pragma unroll
        for (int j = 0; j < kXReq; ++j) request_x(st + 2, xbuf, j);
      } else if (s + kAhead < 4) {
        read_x(s + kAhead, xbuf);
      }
      if constexpr (kDirect)
        if (s == 0 && brings_chunk && !loose) request_chunk(next_chunk, cbuf_now ^ 1);
      if (s == 1) {
#pragma unroll
        for (int j = 0; j < kWReq; ++j) request_w(st + WB, wbuf_now, j);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = mfma32<FP16>(wf[s & 1][t], xf[s & kAhead][i], acc[i][t]);
      if (s == 3) take_scales();
#pragma unroll
      for (int t = 0; t < NT; ++t)
        wf[(s + 1) & 1][t] = dequant8<FP16>(s == 0 ? wc[t].y : s == 1 ? wc[t].z : s == 2 ? wc[t].w : wc[t].x, sc[t], sc16[t], bc[t], mask0, mask4);
      constexpr int kVector = (20 + MT - 1) / MT;
#pragma unroll
      for (int i = 0; i < MT * NT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, kVector, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      // (used in the next step only, the weights would be dequantised there)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        asm volatile("" : "+v"(wf[(s + 1) & 1][t].x), "+v"(wf[(s + 1) & 1][t].y), "+v"(wf[(s + 1) & 1][t].z), "+v"(wf[(s + 1) & 1][t].w));
      if (s == 2) read_codes();
    }
    xbuf ^= 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the requests that nobody reads: LDS is used for other things, or the workgroup leaves

  auto mine = [&](int i) __attribute__((always_inline)) { return KG == 1 || i % KG == kg; };
  if constexpr (KG > 1) {
    // Row of tiles i is finished by set i % KG: the others hand their sums over through LDS, as many rows of tiles at a
    // time as fit the stages.
    constexpr int kRow = (KG - 1) * NT * 4 * kSet;  // 16-byte pieces that are handed over for a row of tiles
    constexpr int kPer = T::kFrontBytes / (16 * kRow) < MT ? T::kFrontBytes / (16 * kRow) : MT;
    static_assert(kPer > 0, "the stages hold the sums of a row of tiles");
    f32x4_t* const red = reinterpret_cast<f32x4_t*>(lds) + tid % kSet;
    __syncthreads();
#pragma unroll
    for (int i0 = 0; i0 < MT; i0 += kPer) {
      if (i0 > 0) __syncthreads();
#pragma unroll
      for (int i = i0; i < i0 + kPer && i < MT; ++i) {
        if (mine(i)) continue;
        f32x4_t* const to = red + (i - i0) * kRow + (kg - (kg > i % KG ? 1 : 0)) * (NT * 4 * kSet);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            to[(4 * t + q) * kSet] = f32x4_t{acc[i][t][4 * q], acc[i][t][4 * q + 1], acc[i][t][4 * q + 2], acc[i][t][4 * q + 3]};
      }
      __syncthreads();
#pragma unroll
      for (int i = i0; i < i0 + kPer && i < MT; ++i) {
        if (!mine(i)) continue;
#pragma unroll
        for (int o = 0; o < KG - 1; ++o)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x4_t v = red[(i - i0) * kRow + ((o * NT + t) * 4 + q) * kSet];
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[i][t][4 * q + r] += v[r];
            }
      }
    }
  }

  // accumulator r of lane (lr, kq), tile (i, t): row m0 + 32 i + lr, column 16 kq + r of the tile; the tiles of one piece of the
  // result: one, or those of gate and up
  constexpr int kTiles = SILU_MUL ? NT : 1, kUnits = MT * NT / kTiles;
  auto emit = [&](int i, int t, const f32x4_t (&v)[kTiles][4]) __attribute__((always_inline)) {
    const int m = m0 + 32 * i + lr, n = (SILU_MUL ? n0 / 2 + wave * 32 : n0 + (wave * NT + t) * 32) + 16 * kq;
    if (m >= a.M || n >= out_cols) return;
    uint32_t w[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      float o[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = 2 * p + h;
        o[h] = v[0][r >> 2][r & 3];
        if constexpr (SILU_MUL) {
          const float g = round16<FP16>(o[h]), u = round16<FP16>(v[kTiles - 1][r >> 2][r & 3]);
          const float sg = round16<FP16>(sigmoid_of_half(g));
          o[h] = round16<FP16>(g * sg) * u;
        }
      }
      w[p] = pack2<FP16>(o[0], o[1]);
    }
    struct __attribute__((packed, aligned(8))) Loose { uint32_t w[4]; };  // (y starts on 8 bytes)
    Loose* const dst = reinterpret_cast<Loose*>(a.y + (size_t)m * out_cols + n);
    dst[0] = Loose{{w[0], w[1], w[2], w[3]}};
    dst[1] = Loose{{w[4], w[5], w[6], w[7]}};
  };
  if (slices == 1) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (!mine(i)) continue;
#pragma unroll
      for (int t0 = 0; t0 < NT; t0 += kTiles) {
        f32x4_t v[kTiles][4];
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[t][q][r] = acc[i][t0 + t][4 * q + r];
        emit(i, t0, v);
      }
    }
    return;
  }
  // Partial tiles are written through to and read from the level all XCDs share (sc1, as in the streaming kernel).
  constexpr size_t kTileFloats = (size_t)BM * BN;
  float* const first = a.partials + (size_t)cut_tile * slices * kTileFloats;
  float* const part_of = first + slice * kTileFloats + (tid % kSet) * 4;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (!mine(i)) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        stream::store_partial(part_of + ((i * NT + t) * 4 + q) * (4 * kSet),
                              f32x4_t{acc[i][t][4 * q], acc[i][t][4 * q + 1], acc[i][t][4 * q + 2], acc[i][t][4 * q + 3]});
  }
  // every wave's stores are acknowledged before the arrival is counted
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  uint32_t* const s_last = reinterpret_cast<uint32_t*>(lds);  // (what was handed over has been read)
  if (tid == 0) *s_last = atomicInc(&a.counters[cut_tile], (uint32_t)(slices - 1)) == (uint32_t)(slices - 1);
  __syncthreads();
  if (!*s_last) return;
  // In order of k, the pieces of the result dealt to the sets; what a thread needs of several slices is asked for before the first
  // is looked at.
  constexpr int kAtOnce = kTiles == 1 || MT == 2 || MT == 3 ? 4 : 2;
  const auto parts = __builtin_amdgcn_make_buffer_rsrc(first, 0, 0x7FFFFFFF, 0x00027000);
#pragma unroll 1
  for (int u = kg; u < kUnits; u += KG) {
    const int i = SILU_MUL ? u : u / NT, t0 = SILU_MUL ? 0 : u % NT;
    f32x4_t sum[kTiles][4];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[t][q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int c0 = 0; c0 < slices; c0 += kAtOnce) {
      f32x4_t v[kAtOnce][kTiles][4];
#pragma unroll
      for (int c = 0; c < kAtOnce; ++c) {
        const int cc = c0 + c < slices ? c0 + c : slices - 1;
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            v[c][t][q] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                parts, (uint32_t)((tid % kSet) * 16 + ((i * NT + t0 + t) * 4 + q) * (16 * kSet) + cc * (kTileFloats * 4)), 0, 16));
      }
#pragma unroll
      for (int c = 0; c < kAtOnce; ++c)
        if (c0 + c < slices) {
#pragma unroll
          for (int t = 0; t < kTiles; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) sum[t][q] += v[c][t][q];
        }
    }
    emit(i, t0, sum);
  }
}

// A tile shape: what it takes, how long a stage takes it, and its kernels.
struct Shape {
  int mt, nt, w, kg, lds;
  int together;        // workgroups that a CU has room for
  double alone, busy;  // us per stage: of one workgroup on a CU, and of each where they share it
  double start;        // us before the first product and behind the last one
  double brief;        // the same of a call of up to kBriefK
  int most;            // slices
  double loose;        // us more where scales come through registers
  const void* kernel[2][3];  // [fp16][plain, scales of the other type, silu-mul]; null: there is none, or it was never the one to take
  int rows() const { return 32 * mt; }
  int columns() const { return 32 * nt * w; }
};
template <int MT, int NT, int W, int KG, bool MIXED = false, bool PLAIN = true>
Shape shape(int together, double alone, double busy, double start, double brief, int most = 16, double loose = 0.0) {
  Shape s{MT, NT, W, KG, Tile<MT, NT, W, KG>::kLdsBytes, together, alone, busy, start, brief, most, loose, {}};
  if constexpr (PLAIN) {
    s.kernel[0][0] = (const void*)qmm_rows_kernel<false, false, MT, NT, W, KG, false>;
    s.kernel[1][0] = (const void*)qmm_rows_kernel<true, true, MT, NT, W, KG, false>;
  }
  if constexpr (MIXED) {
    s.kernel[0][1] = (const void*)qmm_rows_kernel<false, true, MT, NT, W, KG, false>;
    s.kernel[1][1] = (const void*)qmm_rows_kernel<true, false, MT, NT, W, KG, false>;
  }
  if constexpr (NT == 2) {
    s.kernel[0][2] = (const void*)qmm_rows_kernel<false, false, MT, NT, W, KG, true>;
    s.kernel[1][2] = (const void*)qmm_rows_kernel<true, true, MT, NT, W, KG, true>;
  }
  return s;
}
// (1,1,4,2), (2,1,4,2), (3,1,4,2), (4,1,4,2), (2,2,2,2), (2,2,4,2), (3,2,4,1), (2,2,8,1) and (4,2,8,1) were measured as well:
// without them the best of the rest is 0.3 % slower on average.  The last four, of four waves side by side along K, start and end sooner
// than eight waves do, which is most of a call of few rows and weights (20 rows, us, without / with them: 1024 x 1024 6.5 / 5.7, 3072 x 1024
// 8.6 / 7.7, with the activation 1024 x 6144 9.0 / 7.3; 40 rows 9.5 / 8.0 and 10.5 / 7.6).
constexpr int kShapes = 18;
const Shape* shapes() {
  static const Shape all[kShapes] = {
      shape<1, 1, 1, 8>(1, 0.597, 0.571, 4.87, 4.74, 16, 0.17), shape<2, 1, 1, 8>(1, 0.908, 0.454, 5.30, 5.51),
      shape<1, 1, 2, 4, true>(2, 0.559, 0.472, 3.63, 4.33, 16, 2.02), shape<2, 1, 2, 4>(1, 0.695, 0.447, 3.67, 4.81, 16, 1.08),
      shape<3, 1, 2, 4>(1, 0.860, 0.307, 4.55, 5.32, 16, 1.8), shape<1, 2, 2, 4>(1, 0.984, 0.508, 3.75, 5.05, 16, 1.14),
      shape<2, 2, 2, 4, true>(1, 1.105, 0.401, 4.86, 5.96, 16, 0.81), shape<3, 2, 2, 4>(1, 1.415, 0.390, 5.17, 6.86),
      shape<1, 2, 4, 2>(2, 0.902, 0.767, 3.81, 4.77, 16, 0.75), shape<3, 2, 4, 2>(1, 1.269, 0.363, 5.50, 6.39),
      shape<4, 2, 4, 2, true>(1, 1.469, 0.524, 6.60, 7.93), shape<4, 2, 2, 2>(1, 0.925, 0.546, 3.81, 5.77),
      shape<2, 2, 4, 1>(2, 0.631, 0.528, 4.78, 4.93), shape<4, 2, 4, 1>(2, 0.880, 0.761, 4.92, 5.68),
      shape<1, 1, 1, 4>(3, 0.451, 0.334, 3.53, 3.89, 6, 0.36), shape<2, 1, 1, 4>(2, 0.607, 0.452, 3.78, 4.35, 6, 0.45),
      shape<1, 2, 1, 4>(2, 0.730, 0.491, 2.86, 4.29, 6, 0.62), shape<2, 2, 1, 4, false, false>(1, 0.805, 0.626, 3.57, 4.95, 6)};
  return all;
}

struct Plan {
  const Shape* shape;
  int whole, slices, tiles_m, tiles, stages, grid;
  size_t workspace;
  // qmm_resident's, where it is expected to take less time: chunks of a wave (0: not taken), slices, workspace
  int resident_chunks, resident_slices;
  size_t resident_workspace;
};

constexpr size_t kCounterBytes = 64 * 1024;
constexpr int kBriefK = 640;

bool covers(int M, int K, int N, int group_size, bool mixed, int epilogue) {
  if (epilogue != DFLASH_QMM_EPILOGUE_NONE && (epilogue != DFLASH_QMM_EPILOGUE_SILU_MUL || mixed || N % 32 != 0)) return false;
  return M > 0 && K > 0 && N > 0 && (group_size == 32 || group_size == 64 || group_size == 128) && K % group_size == 0 &&
         N % 16 == 0;
}

// A row's scales do not start on four bytes, or K does not fill the stages.  (Also where the arrays do not, which a plan does not know.)
bool scales_through_registers(int K, int group_size, int kg) { return (K / group_size) % 2 != 0 || K % (kStageK * kg) != 0; }

// Which tile, how many slices of K: the least of a model of the time, fitted to measured combinations (15 matrices of 1 to 178 M
// weights, 20 to 1024 rows, every shape and number of slices; the 3039 within 30 % of the best of their call: 4.5 % rms, and what it picks of 225 calls
// is within 0.5 % of the best on average, 12 % at worst; 2.0 and 19.5 % with the constants of the loop that met behind a stage's last step).  A workgroup takes
// `alone` for a stage, or `busy` times those that share its CU; a chip that is full runs against its power.  Adding slices up takes trips to
// memory and traffic at 3 TB/s and more.
// What a shape takes more where scales come through registers (`loose`) is fitted to 4600 combinations of 120 calls with such K (odd multiples of
// 128 from 1664 to 11904, 320 to 3072 columns, 16 to 200 rows): what is picked of them is within 1.3 % of the best on average and 10 % at worst, without
// it 7.5 and 26 % (17 rows of 7808 x 1024 in groups of 128 11.4 -> 9.9 us, 64 of 10112 x 320 12.5 -> 11.0, 100 of 11904 x 2048 19.1 -> 17.6).
// Four waves along K with no more than four stages and nothing to add up start sooner than the line through longer calls has it: 64 calls of K up to 1472 within
// 2 % of the best, 4 % without that; and so do eight with one column of tiles each (58 rows of
// 3072 x 4000 in groups of 128 10.9 -> 9.2; 116 calls of layers of 1024 to 5120 columns, 33 to 450 rows: within 0.8 % of the best in the mean).
// Calls of up to kBriefK are a start, an end and a few stages, and the line through longer calls has their starts wrong by -0.1 to 1.8 us, as the shape is
// (300 rows of 640 x 4096 8.7 -> 10.3 us, 450 of 512 x 4096 with the activation 9.0 -> 10.8 when that line was fitted anew): a line of their own, fitted to the whole
// products of 394 such calls, 17 to 1000 rows, 256 to 8640 columns.  What it picks of 260 others is within 0.3 % of the best in the mean and 9 % at worst, by the
// line of longer calls of the 244 first ones 3.8 and 25 %.
// Against the kernel whose waves met behind a stage's last step, 620 calls of layers of 1024 to 5120 columns and of K 256 to 1024, 17 to 1024 rows: 0.96 of its time in
// the mean, 15 of them slower by more than 3 %, 9 % at most (21 rows of 1792 x 1952 in groups of 128 6.8 -> 7.4; 80 of 15488 x 4608 30.0 -> 31.7, 40 of 4096 x 23552 with the
// activation 24.7 -> 26.1: the line has another shape, or the kernel with weights in registers, too fast).  K of 384 and 640, where four waves along K bring their scales
// through registers, up to 6 % (64 rows of 384 x 8192 5.2 -> 5.5).
// Slices only while all of them find room at once.  Of more tiles than that, those of the last, incomplete round may be
// cut, with the tile left as it is (5120 x 34816 over 1024 rows: 1088 tiles, two to a CU, the last 64 in slices, 344 us; uncut 382).
Plan make_plan(int M, int K, int N, int group_size, int cus, bool fp16, bool mixed, bool silu_mul) {
  const int form = silu_mul ? 2 : mixed ? 1 : 0;
  auto ceil_div = [](long long a, long long b) { return (int)((a + b - 1) / b); };
  auto microseconds = [&](const Plan& p) {
    const Shape& sh = *p.shape;
    const int slots = cus * sh.together, parts = p.grid - p.whole;
    auto stretch = [&](int on_a_cu, int stages) {  // workgroups one after the other and beside each other
      const int rounds = ceil_div(on_a_cu, sh.together);
      return rounds * sh.start + stages * std::max(sh.alone * rounds, sh.busy * on_a_cu);
    };
    const int rounds = p.whole / slots;
    const double loops = stretch(rounds * sh.together, p.stages) + stretch(ceil_div(parts, cus), ceil_div(p.stages, p.slices));
    const double full = std::min(1.0, (double)p.grid / cus);
    double us;
    if (K <= kBriefK) {
      const int on_a_cu = rounds * sh.together + ceil_div(parts, cus), in_turn = rounds + ceil_div(ceil_div(parts, cus), sh.together);
      us = sh.brief + 1.95 * (in_turn - 1) + 0.45 * (on_a_cu - in_turn) + 1.08 * (loops - in_turn * sh.start) + 0.65 * full + (silu_mul ? 0.74 : 0.0);
      if (scales_through_registers(K, group_size, sh.kg)) us += 0.16;
    } else {
      us = loops * (1 + 0.17 * (full - 0.5)) + 0.76 + (silu_mul ? 0.84 : 0.0);
      if (scales_through_registers(K, group_size, sh.kg)) us += sh.loose;
    }
    if (K > kBriefK && p.slices == 1 && sh.w == 1 && sh.nt == 1 && (sh.kg == 4 ? p.stages <= 4 : sh.mt == 1)) us -= 0.35;
    const int pieces = silu_mul ? sh.mt : sh.mt * sh.nt, at_once = silu_mul && (sh.mt == 1 || sh.mt == 4) ? 2 : 4;
    if (p.slices > 1)
      us += 0.96 + 0.806 * ceil_div(pieces, sh.kg) * ceil_div(p.slices, at_once) + 0.352 * parts * (sh.rows() * 8.0 * sh.columns()) / 3e6;
    return us;
  };
  Plan best{};
  double best_us = 0.;
  for (int i = 0; i < kShapes; ++i) {
    const Shape& sh = shapes()[i];
    if (sh.kernel[fp16][form] == nullptr) continue;
    Plan p{};
    p.shape = &sh;
    p.tiles_m = ceil_div(M, sh.rows());
    const long long tiles = (long long)p.tiles_m * ceil_div(N, sh.columns());
    if (tiles > 0x7fffffff / 16) continue;
    p.tiles = (int)tiles;
    p.stages = ceil_div(K, kStageK * sh.kg);
    const int slots = cus * sh.together, most = sh.kg == 1 ? 4 : sh.most;
    const int rest = p.tiles % slots;
    for (p.slices = 1; p.slices <= sh.most && p.slices <= p.stages; ++p.slices) {
      const bool all = p.tiles < slots;
      if (p.slices > 1 && (all ? p.tiles * p.slices > slots || p.slices > most : rest == 0 || rest * p.slices > 2 * slots)) break;
      p.whole = p.tiles - rest;
      p.grid = p.whole + rest * p.slices;
      const double us = microseconds(p);
      if (best.grid == 0 || us < best_us) best = p, best_us = us;
    }
  }
  best.workspace = best.slices > 1 ? kCounterBytes + (size_t)(best.grid - best.whole) * best.shape->rows() * best.shape->columns() * sizeof(float) : 0;
  double us = 0.;
  int chunks = 0, slices = 0;
  size_t workspace = 0;
  if (!mixed && qmm_resident_rows_plan(M, K, N, group_size, silu_mul, &chunks, &slices, &us, &workspace) && us < best_us)
    best.resident_chunks = chunks, best.resident_slices = slices, best.resident_workspace = workspace;
  return best;
}

// The last few plans of this thread: a model asks for the same ones over and over.
const Plan& plan(int M, int K, int N, int group_size, int cus, bool fp16, bool mixed, bool silu_mul) {
  struct Entry {
    int M, K, N, cus, flags;
    Plan p;
  };
  static thread_local Entry cache[64] = {};
  const int flags = (group_size << 3) | (fp16 ? 4 : 0) | (mixed ? 2 : 0) | (silu_mul ? 1 : 0);
  Entry& e = cache[((unsigned)M * 2654435761u + (unsigned)K * 40503u + (unsigned)N * 69069u + (unsigned)flags) >> 26];
  if (e.M != M || e.K != K || e.N != N || e.cus != cus || e.flags != flags)
    e = Entry{M, K, N, cus, flags, make_plan(M, K, N, group_size, cus, fp16, mixed, silu_mul)};
  return e.p;
}

}  // namespace rows

}  // namespace dflash

extern "C" size_t dflash_qmm_rows_workspace_bytes(int M, int K, int N, int group_size, int act_dtype, int sb_dtype, int epilogue) {
  using namespace dflash;
  if (!rows::covers(M, K, N, group_size, act_dtype != sb_dtype, epilogue)) return 0;
  const rows::Plan& p = rows::plan(M, K, N, group_size, qmm_stream_grid(), act_dtype == DFLASH_FP16, act_dtype != sb_dtype,
                                   epilogue != DFLASH_QMM_EPILOGUE_NONE);
  return std::max(p.workspace, p.resident_workspace);  // (which of the two kernels it is also depends on where the scales start)
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
  const rows::Plan& p = rows::plan(M, K, N, group_size, qmm_stream_grid(), act_dtype == DFLASH_FP16, mixed, silu_mul);
  const size_t given = workspace ? workspace_bytes : 0;
  // (what a call has to bring does not depend on which of the two kernels it is)
  DFLASH_REQUIRE(given >= p.workspace, DFLASH_ERR_WORKSPACE,
                 "dflash_qmm_rows: workspace of %zu bytes needed, %zu given", p.workspace, given);
  if (p.resident_chunks != 0 && given >= p.resident_workspace && (((uintptr_t)scales | (uintptr_t)biases) % 4) == 0)
    return qmm_resident_rows_launch(x, w_q, scales, biases, y, workspace, M, K, N, group_size, act_dtype, silu_mul, p.resident_chunks,
                                    p.resident_slices, (hipStream_t)stream);
  rows::Args a;
  a.x = (const uint16_t*)x; a.w = w_q; a.scales = (const uint16_t*)scales; a.biases = (const uint16_t*)biases;
  a.y = (uint16_t*)y;
  a.counters = (uint32_t*)workspace;
  a.partials = workspace ? (float*)((char*)workspace + rows::kCounterBytes) : nullptr;
  a.M = M; a.K = K; a.N = N;
  const size_t sb_bytes = (size_t)N * (K / group_size) * 2;
  a.loose = rows::scales_through_registers(K, group_size, p.shape->kg) || (((uintptr_t)scales | (uintptr_t)biases) % 4) != 0 || sb_bytes >= (1ull << 31);
  a.group_shift = group_size == 32 ? 5 : group_size == 64 ? 6 : 7;
  a.tiles_m = p.tiles_m; a.tiles = p.tiles; a.whole = p.whole; a.slices = p.slices; a.stages = p.stages;
  const bool fp16 = act_dtype == DFLASH_FP16;
  const int form = silu_mul ? 2 : mixed ? 1 : 0;
  const void* const fn = p.shape->kernel[fp16][form];
  const int lds_bytes = p.shape->lds;
  static bool attr_set[kMaxDevices][rows::kShapes][2][3] = {};
  const int dev = current_device_slot();
  if (lds_bytes > 48 * 1024) {
    bool& set = attr_set[dev][p.shape - rows::shapes()][fp16][form];
    if (!set || dev == kMaxDevices - 1) {
      DFLASH_HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes));
      set = true;
    }
  }
  void* args[] = {&a};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)p.grid), dim3(64 * p.shape->w * p.shape->kg), args, (size_t)lds_bytes, (hipStream_t)stream));
  return DFLASH_OK;
}
