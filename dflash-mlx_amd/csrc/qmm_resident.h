// Up to 16 rows against a 4-bit matrix, x kept in registers, for gfx950: y[M, N] = x[M, K] dequant(W)[N, K]^T.  The kernel; one
// source per activation type (qmm_resident_bf16.hip, qmm_resident_fp16.hip) holds its instances, qmm_resident.hip the choice.
//
// A product of 16 rows is a stream of weights.  The streaming kernel (qmm_m16_stream.hip) shares each unit of it between eight waves
// that meet at a barrier per 18 KiB; here every wave has its own stream and meets the others once per four tiles:
//  * a wave owns NCH chunks of 128 k, of all rows.  Its part of x stays in registers, read once (a compute unit has 512 KiB of them,
//    x of 16 rows and K = 6144 is 192), and its part of 16 rows of W at a time comes through a ring of LDS that no other wave sees:
//    direct loads, two tiles ahead, no registers and no barriers for them;
//  * loads follow the rows: a load instruction covers runs of NCH * 64 bytes, whole 128-byte lines where NCH and the wave's first chunk are even;
//    else the ends of a run share their lines with the waves beside it.  In matrix-instruction order (16 rows, 64 bytes each) the same loads with
//    nothing else took 24.6 us for 5120 x 34816, in this order 17 - 20; for x (256-byte runs, turned through LDS) 2.2 us of a launch.  LDS takes the pieces in an order without bank conflicts; a row's scales are fetched four bytes a lane;
//  * scales and biases enter in fp32 as before: s * sum x q per group on the vector pipe, the sums of x times the biases of four groups in one
//    16 x 16 x 4 fp32 matrix instruction;
//  * the eight waves' sums meet in LDS, in their order.  Where a wave's chunks would be more than NCH, the K range is cut into slices of
//    whole workgroups: all but the last store their tiles (their own arrival flags, see nonzero_words()), the last adds them in order.
//    Those it waits for wait for nobody and have lower indexes, but workgroups start in order on each XCD only, and another stream's kernel can hold one
//    of them back there: the wait ends once they have had their turn, and spin_limit bounds it.
// us, streaming kernel -> here (16 rows, weights from memory): 4096 x 4096 8.0 -> 6.1, 4096 x 7168 9.5 -> 7.7, 5120 x 5120 9.5 -> 7.4, 5120 x 7168 10.8 -> 9.4,
// 12288 x 4096 12.3 -> 10.6, 17408 x 5120 16.3 -> 16.0, 5120 x 34816 with the activation 26.7 -> 24.7, 4096 x 49152 27.0 -> 23.3 (4.85 TB/s).  Eight waves: with
// twelve or sixteen (fewer chunks each) 5 - 13 % slower; three tiles ahead 7 % slower; arithmetic alone takes 20 of the 25 us.
#pragma once
#include <utility>

#include "qmm_stream_device.h"

namespace dflash {
namespace resident {

using stream::Act;
using stream::lds_void_t;
using stream::u32x2_t;

constexpr int kWaves = 8;
constexpr int kChunk = 128;  // k of a piece of 64 bytes of codes
constexpr int kDepth = 2;    // tiles of a wave's ring
constexpr int kMostSlices = 4;
constexpr uint32_t kPast = 0x80000000u;  // an offset behind every array: reads zeros

struct Args {
  const uint16_t* x;  // [M, K]
  const void* w;      // [N, K/8] words, or (PACKED) the images of qmm_pack_kernel (SILU: of qmm_pack_gate_up_kernel), like scales and biases
  const void* scales;
  const void* biases;
  uint16_t* y;  // [M, N], SILU: [M, N / 2]
  float* partials;  // slices > 1: MT = 1: [N / 16][slices - 1] tiles, zero between calls; else [N / 16][MT][slices] tiles
  uint32_t* status;  // MT = 1: its error word; else a counter per N / 16 and MT, zero between calls
  int M, K, N, slices, spin_limit;
  // what the kernel would otherwise divide for before its first request (0.3 us): workgroups of a slice, tiles of each and how many have one more, and the
  // same for steps of K and waves (a step: 128 k, in groups of 128 twice that, whose scales are a word)
  int lanes, tiles_each, tiles_more, steps_each, steps_more;
};
inline void set_partition(Args& p, int group_size, int cus) {
  const int tiles = p.N / 16, of_slice = cus / p.slices, steps = p.K / (group_size == 128 ? 256 : 128), parts = p.slices * kWaves;
  p.lanes = tiles < of_slice ? tiles : of_slice;
  p.tiles_each = tiles / p.lanes, p.tiles_more = tiles % p.lanes;
  p.steps_each = steps / parts, p.steps_more = steps % parts;
}

template <int GS, int NCH, int MT>
struct Geometry {
  static constexpr int kSlots = MT == 1 ? 4 : 2;      // tiles between two meetings of the waves
  static constexpr int G = kChunk / GS, WPG = 4 / G;  // groups of a chunk, words of a lane per group
  static constexpr int SD = (NCH * G + 1) / 2;        // words of a row's scales, two groups each
  static constexpr int NS = (SD + 3) / 4;             // loads for them
  static constexpr int NB = (NCH * G + 3) / 4;        // fp32 matrix instructions for the biases
  static constexpr int kStage = NCH * 1024 + 2 * NS * 256;
  static constexpr int kLoads = NCH + 2 * NS;
  static constexpr int kSums = kWaves * kDepth * kStage;
  static constexpr int kSumsOfWave = kSlots * MT * 1024;
  static constexpr int kLds = kSums + kWaves * kSumsOfWave;
  static_assert(kLds <= 160 * 1024, "LDS of a compute unit");
};

template <int... I, class F>
__device__ __forceinline__ void each(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {
  each(std::make_integer_sequence<int, N>{}, static_cast<F&&>(f));
}

// LDS by hand: the compiler would wait for all of a wave's direct loads before each access.  A read's registers are written until
// the wait that follows it; nothing may touch them in between (isa_check.py).
template <int OFF>
__device__ __forceinline__ void lds_read(uint32_t at, u32x4_t& v) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(v) : "v"(at), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void lds_read(uint32_t at, u32x2_t& v) {
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=&v"(v) : "v"(at), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void lds_read(uint32_t at, uint32_t& v) {
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=&v"(v) : "v"(at), "n"(OFF) : "memory");
}
template <class V>
__device__ __forceinline__ void lds_write16(uint32_t at, V v) {
  asm volatile("ds_write_b128 %0, %1" ::"v"(at), "v"(v) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 8 codes of a word as numbers offset + q, in the slot order of stream::unpack_codes.  What the offset adds to a sum is taken off again, and the rounding
// error of a sum is that of the numbers it is made of, so the offset has to be small or gone before the groups are added up:
//  * it is taken off inside the matrix instructions, which start from -offset * (sum of x over the group) and not from zero (kStart; four registers per
//    group, a launch takes as long as without, 4 chunks and one tile 0.1 us longer);
//  * groups of 32 have registers for that up to three chunks (four: spilled, 4096 x 24576 with the activation 16.5 -> 23.1 us).  Beyond that bf16 codes go to
//    the top of the mantissa, offset 16, for one more shift per word (1 % of a launch);
//  * fp16: the mantissa has room for codes four bits further up, where the offset is 64 and not 1024.
// Share of results that are not those of fp64 rounded, streaming kernel and here: bf16 5120 x 7168 0.12 and 0.06 %, 5120 x 4096 in groups of 32 0.09 and
// 0.07 %; fp16 6.2 and 0.33 %, in groups of 32 5.2 and 1.1 %.  (Offset 128 and those of all groups in one sum in front of the others: bf16 0.25 and 0.32 %.)
template <bool H16, int GS, int NCH>
struct Codes {
  static constexpr bool kStart = GS != 32 || NCH <= 3;
  static constexpr int kUp = H16 ? 4 : kStart ? 0 : 3;  // bits that the codes move up
  static constexpr uint32_t kMask = 0x000F000Fu << kUp, kMagic = H16 ? 0x54005400u : kStart ? Act<false>::kMagic : 0x41804180u;
  static constexpr float kOffset = H16 ? 64.0f : kStart ? Act<false>::kOffset : 16.0f;
  static constexpr uint32_t kMinusOffset = H16 ? 0xD400D400u : 0xC300C300u;  // twice, in the activation type (kStart)
  static __device__ __forceinline__ uint4 unpack(uint32_t w, uint32_t mask, uint32_t magic) {
    auto at = [&](int bit) { return ((bit > kUp ? w >> (bit - kUp) : w << (kUp - bit)) & mask) | magic; };
    return make_uint4(at(0), at(4), at(8), at(12));
  }
};

// Sums of x over groups: xs[i] for the biases, lane (li, q) group 4 i + q of row li; from[c][g], the products' accumulators of that group: -offset times
// those of rows 4 q + r.  One set of matrix instructions for both: its sums are the same in all sixteen lanes of a q, so each picks the group and row of a lane
// that fetches it from there.
template <bool H16, int GS, int NCH>
__device__ __forceinline__ void sums_of_groups(const uint4 (&x)[NCH][4], int li, int q, float (&xs)[Geometry<GS, NCH, 1>::NB],
                                               f32x4_t (&from)[NCH][Geometry<GS, NCH, 1>::G]) {
  using A = Act<H16>;
  using C4 = Codes<H16, GS, NCH>;
  using L = Geometry<GS, NCH, 1>;
  constexpr uint32_t kBy = C4::kStart ? C4::kMinusOffset : A::kOnes;
  const uint4 by = make_uint4(kBy, kBy, kBy, kBy);
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int g = 0; g < L::G; ++g) {
      f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < L::WPG; ++i) d = C4::kStart ? A::mfma(x[c][g * L::WPG + i], by, d) : A::mfma(by, x[c][g * L::WPG + i], d);
      const int gi = c * L::G + g;
      if constexpr (C4::kStart) {
        from[c][g] = d;
        const float sum = li & 2 ? (li & 1 ? d[3] : d[2]) : (li & 1 ? d[1] : d[0]);
        xs[gi >> 2] = (li >> 2) == (gi & 3) ? sum : (gi & 3) == 0 ? 0.f : xs[gi >> 2];
      } else {
        from[c][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        xs[gi >> 2] = q == (gi & 3) ? d[0] : (gi & 3) == 0 ? 0.f : xs[gi >> 2];
      }
    }
  if constexpr (C4::kStart) {
    const int lane = 16 * (li >> 2) + 4 * q + (li & 3);
#pragma unroll
    for (int i = 0; i < L::NB; ++i) xs[i] = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * lane, __float_as_int(xs[i]))) * (-1.0f / C4::kOffset);
  }
}
// What a row's scale s and bias b multiply its sums of x with
template <class C4>
__device__ __forceinline__ float bias_of(float s, float b) {
  return C4::kStart ? b : __builtin_fmaf(-C4::kOffset, s, b);
}

// Weights of 17 rows and more are rounded to the activation type, as in the any-rows product (qmm_rows.hip says how the codes become numbers)
template <bool H16>
__device__ __forceinline__ uint32_t dequant2(uint32_t w, int p, float s24, float s20, float b, uint32_t mask0, uint32_t mask4) {
  const uint32_t v = p & 1 ? w >> 8 : w;
  const f16x2_t lo = __builtin_bit_cast(f16x2_t, v & mask0), hi = __builtin_bit_cast(f16x2_t, v & mask4);
  return pack_pair<H16 ? DFLASH_FP16 : DFLASH_BF16>(__builtin_fmaf((float)lo[p >> 1], s24, b), __builtin_fmaf((float)hi[p >> 1], s20, b));
}
template <bool H16>
__device__ __forceinline__ uint4 dequant8(uint32_t w, float s24, float s20, float b, uint32_t mask0, uint32_t mask4) {
  return make_uint4(dequant2<H16>(w, 0, s24, s20, b, mask0, mask4), dequant2<H16>(w, 1, s24, s20, b, mask0, mask4),
                    dequant2<H16>(w, 2, s24, s20, b, mask0, mask4), dequant2<H16>(w, 3, s24, s20, b, mask0, mask4));
}

template <int WPG>
struct Words {
  typedef u32x4_t T;
  static __device__ __forceinline__ uint32_t get(const T& v, int i) { return v[i]; }
};
template <>
struct Words<2> {
  typedef u32x2_t T;
  static __device__ __forceinline__ uint32_t get(const T& v, int i) { return v[i]; }
};
template <>
struct Words<1> {
  typedef uint32_t T;
  static __device__ __forceinline__ uint32_t get(const T& v, int) { return v; }
};

// up to three other slices' tiles; their loads overlap
__device__ __forceinline__ void load_partials3(const float* const (&p)[3], f32x4_t (&v)[3]) {
  asm volatile(
      "global_load_dwordx4 %0, %3, off sc1\n"
      "global_load_dwordx4 %1, %4, off sc1\n"
      "global_load_dwordx4 %2, %5, off sc1\n"
      "s_waitcnt vmcnt(0)\n"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2])
      : "v"(p[0]), "v"(p[1]), "v"(p[2])
      : "memory");
}

// H16: activations and scales are fp16, else bf16.  GS: group size.  SILU: W holds the gate rows of an MLP and, behind them, its up rows;
// the rows of a tile are 8 gate rows and the up rows of the same columns, so that lane li + 8 of a finished tile holds what lane li
// multiplies with.
template <bool H16, int GS, int NCH, int MT, bool SILU, bool PACKED>
__device__ __forceinline__ void product(const Args& p) {
  using A = Act<H16>;
  using C4 = Codes<H16, GS, NCH>;
  using L = Geometry<GS, NCH, MT>;
  constexpr int kSlots = L::kSlots;
  constexpr int G = L::G, WPG = L::WPG, NS = L::NS, NB = L::NB;
  extern __shared__ __align__(16) char lds[];  // every wave's ring; then the waves' sums
  const int lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, N = p.N, slices = p.slices, lanes_of_slice = p.lanes;
  int slice = 0, tile = (int)blockIdx.x;
  while (tile >= lanes_of_slice) tile -= lanes_of_slice, ++slice;
  const int first_tile = tile, mine_of_tiles = p.tiles_each + (tile < p.tiles_more ? 1 : 0);
  // the wave's chunks
  constexpr int STEP = GS == 128 ? 2 : 1;
  const int part = slice * kWaves + wave;
  const int first = STEP * (part * p.steps_each + (part < p.steps_more ? part : p.steps_more)), mine = STEP * (p.steps_each + (part < p.steps_more ? 1 : 0));

  const int RB = (N + 127) / 128;
  const uint32_t w_bytes = PACKED ? (uint32_t)RB * (uint32_t)(K / 256) * 16384u : (uint32_t)N * (uint32_t)(K / 2);
  const uint32_t s_bytes = PACKED ? (uint32_t)RB * (uint32_t)(K / 1024) * 4096u : (uint32_t)N * (uint32_t)(K / GS) * 2u;
  const auto w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.w), 0, w_bytes, 0x00027000);
  const auto s_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.scales), 0, s_bytes, 0x00027000);
  const auto b_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.biases), 0, s_bytes, 0x00027000);
  const auto x_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x), 0, (uint32_t)p.M * (uint32_t)K * 2u, 0x00027000);

  // x first (from the weights on, a request waits for theirs): 256 bytes of four rows a load; rows past M and chunks past `mine` are zeros
  u32x4_t xr[MT][NCH][4];
  // (MT = 1: loads of rows that are all absent are left out; the last rows go first, so that what follows a load that may be left out are loads
  // that are not, and a wait for any of them counts those only)  (A token through 5120 x 34816 with silu 25.0 -> 23.7 us,
  // 17408 x 5120 16.3 -> 15.7, 4096 x 24576 with silu 15.0 -> 14.6; 16 rows as before.)
#pragma unroll
  for (int j = 3; j >= 0; --j)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const uint32_t at = (uint32_t)(16 * m + 4 * j + q) * (uint32_t)K * 2u + 256u * (uint32_t)(first + c) + 16u * li;
        if (MT == 1 && j > 0 && p.M <= 4 * j) xr[m][c][j] = u32x4_t{0u, 0u, 0u, 0u};
        else xr[m][c][j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(x_buf, c < mine ? at : kPast, 0, 0));
      }
  __builtin_amdgcn_sched_barrier(0);

  // Where the lanes of a load read.  Load j of a tile fills the wave's granules (16 bytes) 64 j .. 64 j + 63; granule (row, pos) holds piece
  // (pos & 3) ^ (row >> 2) of chunk (pos >> 2) ^ flip(row): 16 rows of one piece are in 16 different quarters of the banks.
  auto flip = [](int row) { return NCH % 4 == 0 ? row & 3 : NCH % 2 == 0 ? (row >> 1) & 1 : 0; };
  uint32_t w_at[NCH], s_at[NS];
  auto row_of = [&](int row) { return SILU ? (uint32_t)((row < 8 ? 0 : N / 2) + (row & 7)) : (uint32_t)row; };
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int granule = 64 * j + lane, row = granule / (4 * NCH), pos = granule % (4 * NCH);
    int c = (pos >> 2) ^ flip(row);
    const int piece = (pos & 3) ^ (row >> 2);
    c = first + (c < mine ? c : mine - 1);  // (chunks past `mine`: some codes, times zeros)
    w_at[j] = PACKED ? (uint32_t)(c >> 1) * 16384u + (row >> 3) * (SILU ? 8192 : 1024) + (row & 7) * 128 + 16u * ((4 * (c & 1) + piece) ^ (((row >> 1) & 3) << 1))
                     : row_of(row) * (uint32_t)(K / 2) + 64u * c + 16u * piece;
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) {  // word 4 j + lane % 4 of row lane / 4
    int word = 4 * j + (lane & 3);
    const int last = mine * G / 2 - 1;
    word = word < last ? word : last;
    const int c = first + word;  // (packed: groups of 64, a word is a chunk's)
    s_at[j] = PACKED ? (uint32_t)(c >> 3) * 4096u + 4u * (c & 7) + (SILU ? 2048u * (lane >> 5) + 32u * ((lane >> 2) & 7) : 32u * (lane >> 2))
                     : row_of(lane >> 2) * (uint32_t)(K / GS) * 2u + 2u * G * first + 4u * word;
  }
  char* const ring = lds + wave * (kDepth * L::kStage);
  auto load = [&](int tile, int d, uint32_t past) __attribute__((always_inline)) {
    uint32_t w_tile, s_tile;
    if (PACKED) {  // SILU: rows of a block of the image are 64 gate rows, then their up rows
      const int rb = tile >> 3, in_rb = tile & 7;
      w_tile = (uint32_t)rb * (uint32_t)(K / 256) * 16384u + (uint32_t)in_rb * (SILU ? 1024u : 2048u);
      s_tile = (uint32_t)rb * (uint32_t)(K / 1024) * 4096u + (SILU ? (uint32_t)in_rb * 256u : (uint32_t)(in_rb >> 1) * 1024u + (uint32_t)(in_rb & 1) * 512u);
    } else {
      w_tile = (uint32_t)tile * (SILU ? 8u : 16u) * (uint32_t)(K / 2);
      s_tile = (uint32_t)tile * (SILU ? 8u : 16u) * (uint32_t)(K / GS) * 2u;
    }
    char* const at = ring + d * L::kStage;
#pragma unroll
    for (int j = 0; j < NCH; ++j)  // (read once: the non-temporal policy, 1 - 3 % of a launch)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buf, (lds_void_t*)(at + 1024 * j), 16, w_at[j] | past, w_tile, 0, 2);
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(s_buf, (lds_void_t*)(at + 1024 * NCH + 512 * j), 4, s_at[j] | past, s_tile, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_buf, (lds_void_t*)(at + 1024 * NCH + 512 * j + 256), 4, s_at[j] | past, s_tile, 0, 0);
    }
  };
  int left = mine_of_tiles;
#pragma unroll
  for (int d = 0; d < kDepth; ++d) load(d < left ? tile + d * lanes_of_slice : 0, d, d < left ? 0u : kPast);
  __builtin_amdgcn_sched_barrier(0);

  // x to the order of the products, a chunk at a time through the wave's 4 KiB of sums: lane (li, q) has row li, of group g the k
  // from GS / 4 * q on, like the codes it reads
  const uint32_t lds0 = stream::lds_address(lds);
  const uint32_t sums_at = lds0 + L::kSums + wave * L::kSumsOfWave;
  uint4 x[MT][NCH][4];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
#pragma unroll
      for (int j = 0; j < 4; ++j) lds_write16(sums_at + 1024u * j + 256u * q + 16u * (li ^ (4 * j + q)), xr[m][c][j]);
      u32x4_t t[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t piece = (uint32_t)((GS / 8) * (i / WPG) + (GS / 32) * q + i % WPG);
        lds_read<0>(sums_at + 256u * li + 16u * (piece ^ li), t[i]);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3])::"memory");
#pragma unroll
      for (int i = 0; i < 4; ++i) x[m][c][i] = stream::as_uint4(MT == 1 ? stream::permute_x(t[i]) : t[i]);
    }
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  float xs[NB];
  f32x4_t from[NCH][G];
  if constexpr (MT == 1) sums_of_groups<H16, GS, NCH>(x[0], li, q, xs, from);

  // in registers the compiler cannot see through: one v_and_or_b32 per pair of codes, selections without branches
  uint32_t mask = MT == 1 ? C4::kMask : 0x000F000Fu, mask4 = 0x00F000F0u, magic = C4::kMagic, upper = q & 2 ? ~0u : 0u;
  asm("" : "+s"(mask), "+s"(mask4), "+v"(magic), "+v"(upper));
  const uint32_t half = q & 1 ? 0u : 16u;
  auto low = [](uint32_t v) { return H16 ? f16_bits_to_f32(v & 0xFFFFu) : __uint_as_float(v << 16); };
  auto high = [](uint32_t v) { return H16 ? f16_bits_to_f32(v >> 16) : __uint_as_float(v & 0xFFFF0000u); };
  auto of_q = [&](uint32_t lo, uint32_t hi) {  // of the groups in two words, the lane's
    const uint32_t v = (upper & hi) | (~upper & lo);
    return H16 ? f16_bits_to_f32((v >> (16 - half)) & 0xFFFFu) : __uint_as_float((v << half) & 0xFFFF0000u);
  };
  constexpr int CX = NCH % 4 == 0 ? 4 : NCH % 2 == 0 ? 2 : 1;  // chunks whose addresses differ by more than a constant
  const uint32_t ring_at = lds0 + wave * (kDepth * L::kStage);
  uint32_t codes_at[CX][G];
#pragma unroll
  for (int c = 0; c < CX; ++c)
#pragma unroll
    for (int g = 0; g < G; ++g)
      codes_at[c][g] = ring_at + (uint32_t)(64 * NCH * li + 64 * (c ^ flip(li))) +
                       (G == 1   ? 16u * (q ^ (li >> 2))
                        : G == 2 ? 16u * ((2 * g + (q >> 1)) ^ (li >> 2)) + 8u * (q & 1)
                                 : 16u * (g ^ (li >> 2)) + 4u * q);
  const uint32_t scales_at = ring_at + 1024 * NCH + 16 * li;

  auto step = [&](auto stage, int tile, int left, int slot) __attribute__((always_inline)) {
    constexpr int D = decltype(stage)::value;
    if (left > 1) wait_loads<L::kLoads>();
    else wait_loads<0>();
    typename Words<WPG>::T w[NCH][G];
    u32x4_t s[NS], b[NS];
    each<NS>([&](auto j) __attribute__((always_inline)) {
      constexpr int J = decltype(j)::value;
      lds_read<D * L::kStage + 512 * J>(scales_at, s[J]);
      lds_read<D * L::kStage + 512 * J + 256>(scales_at, b[J]);
    });
    each<NCH * G>([&](auto j) __attribute__((always_inline)) {
      constexpr int C = decltype(j)::value / G, GG = decltype(j)::value % G;
      lds_read<D * L::kStage + 64 * (C / CX * CX)>(codes_at[C % CX][GG], w[C][GG]);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < NS; ++j) asm volatile("" : "+v"(s[j]), "+v"(b[j]));
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int g = 0; g < G; ++g) asm volatile("" : "+v"(w[c][g]));
    if (left > kDepth) load(tile + kDepth * lanes_of_slice, D, 0u);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MT == 1) {
      f32x4_t acc = zero;
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const float sv = of_q(s[i >> 1][2 * (i & 1)], s[i >> 1][2 * (i & 1) + 1]);
        const float bv = of_q(b[i >> 1][2 * (i & 1)], b[i >> 1][2 * (i & 1) + 1]);
        acc = mfma4(xs[i], bias_of<C4>(sv, bv), acc);
      }
#pragma unroll
      for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int g = 0; g < G; ++g) {
          f32x4_t d = from[c][g];
#pragma unroll
          for (int i = 0; i < WPG; ++i) d = A::mfma(x[0][c][g * WPG + i], C4::unpack(Words<WPG>::get(w[c][g], i), mask, magic), d);
          const int gi = c * G + g, word = gi >> 1;
          const float sv = gi & 1 ? high(s[word >> 2][word & 3]) : low(s[word >> 2][word & 3]);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf(sv, d[r], acc[r]);
        }
      lds_write16(sums_at + 1024u * slot + 16u * lane, acc);
    } else {  // weights rounded to the activation type
      f32x4_t acc[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m] = zero;
#pragma unroll
      for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int gi = c * G + g, word = gi >> 1;
          const uint32_t sw = s[word >> 2][word & 3], bw = b[word >> 2][word & 3];
          const float sv = gi & 1 ? high(sw) : low(sw), bv = gi & 1 ? high(bw) : low(bw), s24 = sv * 0x1p24f, s20 = sv * 0x1p20f;
#pragma unroll
          for (int i = 0; i < WPG; ++i) {
            const uint4 v = dequant8<H16>(Words<WPG>::get(w[c][g], i), s24, s20, bv, mask, mask4);
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = A::mfma(x[m][c][g * WPG + i], v, acc[m]);
          }
        }
      // the wait states between a matrix instruction and a store of its result: the compiler does not see the stores inside their blocks
#pragma unroll
      for (int m = 0; m < MT; ++m) asm volatile("" : "+v"(acc[m]));
      asm volatile("s_nop 7\n s_nop 7\n s_nop 7" ::: "memory");
#pragma unroll
      for (int m = 0; m < MT; ++m) lds_write16(sums_at + 1024u * (slot * MT + m) + 16u * lane, acc[m]);
    }
  };

  // The waves deal out the 16 x 16 pieces of the last `count` tiles, add them up and store them
  const int cols = SILU ? N >> 1 : N;
  auto emit = [&](int t, int row0, f32x4_t sum, bool mine_to_store) __attribute__((always_inline)) {
    const int n = (SILU ? 8 : 16) * t + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = sum[r];
      if (SILU) {  // lane li of 16 reads lane li ^ 8 (DPP row_ror:8)
        const float up = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false));
        v = stream::silu_mul<H16>(v, up);
      }
      if (mine_to_store && (!SILU || li < 8) && row0 + 4 * q + r < p.M) p.y[(size_t)(row0 + 4 * q + r) * cols + n] = (uint16_t)A::from_f32(v);
    }
  };
  auto finish = [&](int base, int count, bool more) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int unit = wave; unit < count * MT; unit += kWaves) {
      const int t = base + unit / MT * lanes_of_slice, row0 = MT == 1 ? 0 : 16 * (unit % MT);
      f32x4_t sum;
#pragma unroll
      for (int v0 = 0; v0 < kWaves; v0 += 4) {
        u32x4_t v[4];
        each<4>([&](auto i) __attribute__((always_inline)) {
          constexpr int I = decltype(i)::value;
          lds_read<I * L::kSumsOfWave>(lds0 + L::kSums + v0 * L::kSumsOfWave + 1024u * unit + 16u * lane, v[I]);
        });
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])::"memory");
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4_t f = __builtin_bit_cast(f32x4_t, v[i]);
          sum = v0 + i == 0 ? f : sum + f;
        }
      }
      bool mine_to_store = true;
      if (MT == 1 && slices > 1) {
        float* const slot = p.partials + ((size_t)t * (slices - 1) * 64 + lane) * 4;
        if (slice < slices - 1) {
          stream::store_partial(slot + slice * 256, stream::nonzero_words(sum));
          mine_to_store = false;
        } else {
          f32x4_t total = zero;
          for (int s0 = 0; s0 < slices - 1; s0 += 3) {
            const float* src[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) src[i] = slot + (s0 + i < slices - 1 ? s0 + i : slices - 2) * 256;  // (surplus ones: the last again)
            f32x4_t v[3];
            for (int polls = 0;;) {
              load_partials3(src, v);
              uint32_t present = 1u;
#pragma unroll
              for (int i = 0; i < 3; ++i) {
                const u32x4_t bits = __builtin_bit_cast(u32x4_t, v[i]);
                present = min(present, min(min(bits.x, bits.y), min(bits.z, bits.w)));
              }
              if (__builtin_amdgcn_ballot_w64(present == 0u) == 0ull) break;
              if (++polls > p.spin_limit) {
                // gives up: the launch ends, these rows are wrong, and the caller can tell
                if (lane == 0)
                  __hip_atomic_store(&p.status[stream::kErrorWord], 0x80000000u | (uint32_t)(t >> 3), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
              }
              __builtin_amdgcn_s_sleep(2);
            }
#pragma unroll
            for (int i = 0; i < 3; ++i)
              if (s0 + i < slices - 1) {
                total += v[i];
                stream::store_partial(const_cast<float*>(src[i]), zero);
              }
          }
          sum = total + sum;
        }
      }
      if (MT > 1 && slices > 1) {
        stream::store_partial(p.partials + ((size_t)((t * MT + unit % MT) * slices + slice) * 64 + lane) * 4, sum);
        continue;
      }
      emit(t, row0, sum, mine_to_store);
    }
    if (more) asm volatile("s_barrier" ::: "memory");
  };

  int base = tile, slot = 0;
  for (; left >= kDepth; left -= kDepth) {
    each<kDepth>([&](auto d) __attribute__((always_inline)) {
      step(d, tile, left - decltype(d)::value, slot + decltype(d)::value);
      tile += lanes_of_slice;
    });
    slot += kDepth;
    if (slot + kDepth > kSlots && left > kDepth) {
      finish(base, slot, true);
      base = tile, slot = 0;
    }
  }
  if (left > 0) step(std::integral_constant<int, 0>{}, tile, left, slot++);
  finish(base, slot, false);
  if (MT > 1 && slices > 1) {
    // The last slice to come to its tiles adds up what all have stored, in order; nobody waits.  (A slice's stores are acknowledged
    // before it says so.)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    uint32_t before = 0;
    if (lane == 0 && wave == 0) before = atomicInc(&p.status[first_tile], (uint32_t)(slices - 1));
    if (wave == 0) {
      const uint32_t told = __builtin_amdgcn_readfirstlane(before);
      asm volatile("ds_write_b32 %0, %1\n s_waitcnt lgkmcnt(0)" ::"v"(lds0), "v"(told) : "memory");
    }
    asm volatile("s_barrier" ::: "memory");
    if ((int)stream::lds_read_u32(lds0) != slices - 1) return;
    for (int unit = wave; unit < mine_of_tiles * MT; unit += kWaves) {
      const int t = first_tile + unit / MT * lanes_of_slice, m = unit % MT;
      float* const slot_of = p.partials + ((size_t)((t * MT + m) * slices) * 64 + lane) * 4;
      f32x4_t total = zero;
      for (int s0 = 0; s0 < slices; s0 += 3) {
        const float* src[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) src[i] = slot_of + (s0 + i < slices ? s0 + i : slices - 1) * 256;
        f32x4_t v[3];
        load_partials3(src, v);
#pragma unroll
        for (int i = 0; i < 3; ++i)
          if (s0 + i < slices) total += v[i];
      }
      emit(t, 16 * m, total, true);
    }
  }
}

template <bool H16, int GS, int NCH, int MT, bool SILU, bool PACKED>
__global__ __launch_bounds__(64 * kWaves, 2) void qmm_resident_kernel(Args p) {
  product<H16, GS, NCH, MT, SILU, PACKED>(p);
}

// The instance for a shape and its LDS; null where there is none.
struct Kernel {
  const void* fn;
  int lds;
};
template <bool H16, int GS, int NCH, int MT, bool PACKED>
Kernel kernel_of(bool silu) {
  const void* fn = silu ? (const void*)qmm_resident_kernel<H16, GS, NCH, MT, true, PACKED> : (const void*)qmm_resident_kernel<H16, GS, NCH, MT, false, PACKED>;
  return {fn, Geometry<GS, NCH, MT>::kLds};
}
// Most chunks that the registers hold: x takes 16 per chunk and 16 rows.
constexpr int most_chunks(int group_size, int row_tiles) {
  return row_tiles == 1 ? (group_size == 32 ? 5 : 6) : row_tiles == 2 ? (group_size == 128 ? 4 : 5) : row_tiles == 3 ? (group_size == 128 ? 2 : 3) : 2;
}
template <bool H16, int GS, int MT, bool PACKED>
Kernel kernel_of(int chunks, bool silu) {
  constexpr int most = most_chunks(GS, MT);
  if (chunks == 2) return kernel_of<H16, GS, 2, MT, PACKED>(silu);
  if constexpr (most >= 4) {
    if (chunks == 4) return kernel_of<H16, GS, 4, MT, PACKED>(silu);
  }
  if constexpr (most >= 6) {
    if (chunks == 6) return kernel_of<H16, GS, 6, MT, PACKED>(silu);
  }
  if constexpr (GS != 128 && most >= 3) {
    if (chunks == 3) return kernel_of<H16, GS, 3, MT, PACKED>(silu);
  }
  if constexpr (GS != 128 && most >= 5) {
    if (chunks == 5) return kernel_of<H16, GS, 5, MT, PACKED>(silu);
  }
  return {nullptr, 0};
}
template <bool H16, int MT>
Kernel kernel_of(int group_size, int chunks, bool silu) {
  return group_size == 32 ? kernel_of<H16, 32, MT, false>(chunks, silu)
         : group_size == 64 ? kernel_of<H16, 64, MT, false>(chunks, silu)
                            : kernel_of<H16, 128, MT, false>(chunks, silu);
}
template <bool H16>
Kernel few_kernel(int group_size, int chunks, bool silu, bool packed) {
  return packed ? kernel_of<H16, 64, 1, true>(chunks, silu) : kernel_of<H16, 1>(group_size, chunks, silu);
}
template <bool H16>
Kernel rows_kernel(int row_tiles, int group_size, int chunks, bool silu) {
  switch (row_tiles) {
    case 2: return kernel_of<H16, 2>(group_size, chunks, silu);
    case 3: return kernel_of<H16, 3>(group_size, chunks, silu);
    case 4: return kernel_of<H16, 4>(group_size, chunks, silu);
    case 5: return kernel_of<H16, 5>(group_size, chunks, silu);
    default: return {nullptr, 0};
  }
}
constexpr int kMostRowTiles = 5;
Kernel bf16_kernel(int group_size, int chunks, bool silu, bool packed);
Kernel fp16_kernel(int group_size, int chunks, bool silu, bool packed);
Kernel bf16_rows_kernel(int row_tiles, int group_size, int chunks, bool silu);  // 16 * row_tiles rows
Kernel fp16_rows_kernel(int row_tiles, int group_size, int chunks, bool silu);

}  // namespace resident
}  // namespace dflash
