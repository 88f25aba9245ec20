// Up to 16 rows against a 4-bit matrix of few weights, for gfx950: y[M, N] = x[M, K] dequant(W)[N, K]^T.
//
// The streaming kernel (qmm_m16_stream.hip) gives every compute unit the same share of the weights, units of 128 rows and 256
// columns, and pays for it around the stream: the first unit goes through LDS before a wave has anything to do, and the
// partial sums of a row block meet through memory, 4 us of a launch together.  A matrix that is a unit or two for each
// compute unit is nothing but these costs.  Here a workgroup has 16 (or 32) rows of W and all of K, so that no sum leaves
// it:
//  * a wave takes every eighth 128 columns; a lane's 16 bytes of codes go from memory to the registers that multiply them, four
//    such loads in flight per wave, and with eight waves all of a K of 4096 is asked for before anything is looked at;
//  * a lane has 32 consecutive codes, but a matrix instruction has to stay within a group: the halves of the wave (groups of 64) or
//    all four lane groups (32) exchange registers, two or four v_permlane swaps, and x is read in the order that follows;
//  * x goes through LDS (rows 16 bytes longer than K, so that the 16 rows of a read are in different banks): asked for by each wave where it multiplies, it
//    was 64 of the 100 cycles that the address units spend on 128 columns;
//  * sums of the eight waves meet in LDS, in their order.  Which rows come along changes nothing: a row has the same bits alone.
// us, streaming kernel -> here, one row / 16 rows: 1024 x 512 5.8 -> 3.3 / 6.1 -> 3.9;  2304 x 3200 7.5 -> 3.9 / 7.7 -> 5.8;
// 3584 x 4096 7.2 -> 4.9 / 7.5 -> 7.2;  4736 x 2304 9.0 -> 6.0 / 9.4 -> 8.4;  groups of 32, 1280 x 1792 6.6 -> 3.4 / 6.9 -> 4.3.
// What bounds it now: the launch, one trip to memory, and with 16 rows x, which every compute unit fetches for itself
// (2304: 74 KB against 18 KB of weights).
#include "qmm_stream_device.h"

namespace dflash {
namespace narrow {
namespace {

using stream::Act;
using stream::u32x2_t;

constexpr int kWaves = 8;
constexpr int kBatch = 4;    // chunks a wave asks for at a time
constexpr int kChunk = 128;  // k of one weight load: 16 bytes of each of 16 rows per four lanes

struct Args {
  const uint16_t* x;  // [M, K]
  const void* w;      // [N, K/8] words, or (PACKED) the images of qmm_pack_kernel, like scales and biases
  const void* scales;
  const void* biases;
  uint16_t* y;  // [M, N], SILU: [M, N / 2]
  int M, K, N;
};

__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {  // a of lanes 32 .. 63 with b of lanes 0 .. 31
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0], b = r[1];
}
__device__ __forceinline__ void swap_rows(uint32_t& a, uint32_t& b) {  // a of lanes 16 .. 31, 48 .. 63 with b of lanes 0 .. 15, 32 .. 47
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0], b = r[1];
}

template <int GS, int NT>
struct Chunk {
  u32x4_t w[NT];
  u32x2_t s[NT], b[NT];  // the scales and biases of the chunk's groups (low halves first)
};

// NT: tiles of 16 rows of W.  SILU: W holds the gate rows of an MLP and, behind them, its up rows; the rows of a tile are 8 gate rows
// and the up rows of the same columns, so that lane li + 8 of a finished tile holds what lane li multiplies with.
template <bool A16, bool S16, int GS, int NT, bool SILU, bool PACKED>
__global__ __launch_bounds__(64 * kWaves) void qmm_narrow_kernel(Args p) {
  constexpr int W = kWaves;
  using A = Act<A16>;
  constexpr int G = kChunk / GS, WPG = 4 / G;  // groups of a chunk, words of a lane per group
  extern __shared__ __align__(16) char lds[];  // x, rows of 2 K + 16 bytes; then the waves' sums
  const int lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, N = p.N, chunks = K / kChunk;
  const int col0 = blockIdx.x * (SILU ? 8 * NT : 16 * NT);
  const int RB = (N + 127) / 128;
  const uint32_t w_bytes = PACKED ? (uint32_t)RB * (K / 256) * 16384u : (uint32_t)N * (uint32_t)(K / 2);
  const uint32_t s_bytes = PACKED ? (uint32_t)RB * (K / 1024) * 4096u : (uint32_t)N * (uint32_t)(K / GS) * 2u;
  const auto w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.w), 0, w_bytes, 0x00027000);
  const auto s_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.scales), 0, s_bytes, 0x00027000);
  const auto b_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.biases), 0, s_bytes, 0x00027000);
  const auto x_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x), 0, (uint32_t)p.M * (uint32_t)K * 2u, 0x00027000);
  // x to LDS: its requests first, those of the weights behind them
  const int pieces_of_row = K >> 3, pieces = p.M * pieces_of_row, pitch = 2 * K + 16;

  // Lane (li, q): row li of each tile of the matrix, 16 bytes at 16 q of the chunk's 64 per row
  uint32_t w_at[NT], s_at[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int row = SILU ? (li < 8 ? 0 : N / 2) + col0 + 8 * t + (li & 7) : col0 + 16 * t + li;
    if (PACKED) {
      const int rb = row >> 7, v = row & 127;
      w_at[t] = (uint32_t)rb * (K / 256) * 16384u + (v >> 3) * 1024 + (v & 7) * 128;  // (granules within the row: by chunk)
      s_at[t] = (uint32_t)rb * (K / 1024) * 4096u + (v >> 5) * 1024 + (v & 31) * 32;
    } else {
      w_at[t] = (uint32_t)row * (uint32_t)(K / 2) + 16 * q;
      s_at[t] = (uint32_t)row * (uint32_t)(K / GS) * 2u;
    }
  }
  const int x_row = li < p.M ? li : p.M - 1;  // (rows past M: some row, their sums are not stored)
  const uint32_t x_at = (uint32_t)(x_row * pitch) + 2u * (GS == 128 ? 32 * q : GS == 64 ? 32 * (q & 1) + 16 * (q >> 1) : 8 * q);
  const int swizzle = ((li >> 1) & 3) << 1;  // (of the packed images; rows of a tile start at a multiple of eight)

  auto load = [&](int j, Chunk<GS, NT>& c) __attribute__((always_inline)) {
    const uint32_t past = j < chunks ? 0u : 0x80000000u;  // chunks that are not there read zeros
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t at = PACKED ? w_at[t] + (uint32_t)(j >> 1) * 16384u + 16u * ((4 * (j & 1) + q) ^ swizzle) : w_at[t] + 64u * j;
      c.w[t] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_buf, at | past, 0, 0));
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t at = PACKED ? s_at[t] + (uint32_t)(j >> 3) * 4096u + 4u * (j & 7) : s_at[t] + 2u * G * j;
      if (GS == 32) {
        c.s[t] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(s_buf, at | past, 0, 0));
        c.b[t] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(b_buf, at | past, 0, 0));
      } else if (GS == 64) {
        c.s[t][0] = __builtin_amdgcn_raw_buffer_load_b32(s_buf, at | past, 0, 0);
        c.b[t][0] = __builtin_amdgcn_raw_buffer_load_b32(b_buf, at | past, 0, 0);
      } else {
        c.s[t][0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(s_buf, at | past, 0, 0);
        c.b[t][0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(b_buf, at | past, 0, 0);
      }
    }
  };

  f32x4_t acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const uint4 ones = make_uint4(A::kOnes, A::kOnes, A::kOnes, A::kOnes);
  uint32_t mask = 0x000F000Fu, magic = A::kMagic;  // in registers the compiler cannot see through: one v_and_or_b32 per pair of codes
  asm("" : "+s"(mask), "+v"(magic));
  auto multiply = [&](int j, Chunk<GS, NT>& c) __attribute__((always_inline)) {
    uint4 a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      a[i] = stream::as_uint4(stream::permute_x(*reinterpret_cast<const u32x4_t*>(lds + x_at + 2u * (kChunk * j + GS * (i / WPG) + 8 * (i % WPG)))));
#pragma unroll
    for (int t = 0; t < NT; ++t) {  // word i of a lane: 8 codes of group i / WPG, like its x
      uint32_t w0 = c.w[t][0], w1 = c.w[t][1], w2 = c.w[t][2], w3 = c.w[t][3];
      if (GS < 128) swap_halves(w0, w2), swap_halves(w1, w3);
      if (GS == 32) swap_rows(w0, w1), swap_rows(w2, w3);
      c.w[t] = u32x4_t{w0, w1, w2, w3};
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      f32x4_t xs = zero;
#pragma unroll
      for (int i = 0; i < WPG; ++i) xs = A::mfma(a[g * WPG + i], ones, xs);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        f32x4_t d = zero;
#pragma unroll
        for (int i = 0; i < WPG; ++i) d = A::mfma(a[g * WPG + i], stream::unpack_codes(c.w[t][g * WPG + i], mask, magic), d);
        const uint32_t sw = c.s[t][g >> 1], bw = c.b[t][g >> 1];
        const float s = S16 ? f16_bits_to_f32(g & 1 ? sw >> 16 : sw & 0xFFFFu) : __uint_as_float(g & 1 ? sw & 0xFFFF0000u : sw << 16);
        const float b = S16 ? f16_bits_to_f32(g & 1 ? bw >> 16 : bw & 0xFFFFu) : __uint_as_float(g & 1 ? bw & 0xFFFF0000u : bw << 16);
        const float bb = __builtin_fmaf(-A::kOffset, s, b);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t][r] = __builtin_fmaf(bb, xs[r], __builtin_fmaf(s, d[r], acc[t][r]));
      }
    }
  };

  Chunk<GS, NT> cur[kBatch], nxt[kBatch];
  auto load_batch = [&](int j, Chunk<GS, NT> (&c)[kBatch]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) load(j + i * W, c[i]);
    __builtin_amdgcn_sched_barrier(0xF);
  };
  auto stage = [&](int piece, u32x4_t v) __attribute__((always_inline)) {
    const int row = piece / pieces_of_row, at = piece - row * pieces_of_row;
    if (piece < pieces) *reinterpret_cast<u32x4_t*>(lds + row * pitch + 16 * at) = v;
  };
  auto x_piece = [&](int piece) __attribute__((always_inline)) {
    return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(x_buf, 16u * (uint32_t)piece, 0, 0));
  };
  int j = wave;
  if (pieces <= 64 * W) {
    const u32x4_t v = x_piece(threadIdx.x);
    load_batch(j, cur);
    stage(threadIdx.x, v);
  } else {
    constexpr int kPieces = 8;
    u32x4_t v[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) v[i] = x_piece(threadIdx.x + 64 * W * i);
    load_batch(j, cur);
#pragma unroll
    for (int i = 0; i < kPieces; ++i) stage(threadIdx.x + 64 * W * i, v[i]);
    for (int base = 64 * W * kPieces; base < pieces; base += 64 * W * kPieces) {
#pragma unroll
      for (int i = 0; i < kPieces; ++i) v[i] = x_piece(base + threadIdx.x + 64 * W * i);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) stage(base + threadIdx.x + 64 * W * i, v[i]);
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  for (; j + kBatch * W < chunks; j += kBatch * W) {
    load_batch(j + kBatch * W, nxt);
#pragma unroll
    for (int i = 0; i < kBatch; ++i) multiply(j + i * W, cur[i]);
#pragma unroll
    for (int i = 0; i < kBatch; ++i) cur[i] = nxt[i];
  }
#pragma unroll
  for (int i = 0; i < kBatch; ++i)
    if (j + i * W < chunks) multiply(j + i * W, cur[i]);
  __syncthreads();
  f32x4_t* const red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
  for (int t = 0; t < NT; ++t) red[(wave * NT + t) * 64 + lane] = acc[t];
  __syncthreads();
  if (wave >= NT) return;
  f32x4_t sum = red[wave * 64 + lane];
#pragma unroll
  for (int w = 1; w < W; ++w) sum += red[(w * NT + wave) * 64 + lane];
  const int cols = SILU ? N >> 1 : N, n = col0 + (SILU ? 8 : 16) * wave + li;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v = sum[r];
    if (SILU) {  // lane li of 16 reads lane li ^ 8 (DPP row_ror:8)
      const float up = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false));
      v = stream::silu_mul<A16>(v, up);
    }
    if ((!SILU || li < 8) && 4 * q + r < p.M) p.y[(size_t)(4 * q + r) * cols + n] = (uint16_t)A::from_f32(v);
  }
}

template <bool A16, bool S16, int NT>
const void* kernel_for(int GS, bool silu, bool packed) {
  if (packed) return (const void*)qmm_narrow_kernel<A16, S16, 64, NT, false, true>;
  if (silu)  // (one type for activations and scales)
    return GS == 32 ? (const void*)qmm_narrow_kernel<A16, A16, 32, NT, true, false>
           : GS == 64 ? (const void*)qmm_narrow_kernel<A16, A16, 64, NT, true, false>
                      : (const void*)qmm_narrow_kernel<A16, A16, 128, NT, true, false>;
  return GS == 32 ? (const void*)qmm_narrow_kernel<A16, S16, 32, NT, false, false>
         : GS == 64 ? (const void*)qmm_narrow_kernel<A16, S16, 64, NT, false, false>
                    : (const void*)qmm_narrow_kernel<A16, S16, 128, NT, false, false>;
}
template <int NT>
const void* kernel_for(bool a16, bool s16, int GS, bool silu, bool packed) {
  return a16 ? (s16 ? kernel_for<true, true, NT>(GS, silu, packed) : kernel_for<true, false, NT>(GS, silu, packed))
             : (s16 ? kernel_for<false, true, NT>(GS, silu, packed) : kernel_for<false, false, NT>(GS, silu, packed));
}

// Tiles of a workgroup, 0: not this kernel's.  One round of workgroups on 256 compute units: 16 rows of W each up to N = 4096; 32 each up to
// 8192, where a K of 2048 is the last that 16 rows of x do not make slower (2048 x 8192 7.5 -> 7.0 us, 2560 x 6144 7.5 -> 7.8).
// Beyond K = 3584 x alone takes as long as the partial sums did (4096 x 4096, 16 rows: 7.9 -> 8.3 us, one row 7.6 -> 6.0), except
// where the streaming kernel cuts few row blocks into many (4736 x 2304 9.4 -> 8.4; 4096 x 2048, 8.6 against 7.9, is still the
// streaming kernel's).  K below 512 is the tile kernel's (256 x 512: 2.65 us, here 2.66).  M does not enter: a row must not change
// with the rows beside it.
int tiles_for(int K, int N, int group_size) {
  if ((group_size != 32 && group_size != 64 && group_size != 128) || K % kChunk != 0 || N % 16 != 0 || K < 512 || N < 16) return 0;
  if (N <= 4096 && (K <= 3584 || (K <= 4864 && K != 4096 && N <= 2304))) return 1;
  return N <= 8192 && K <= 2048 && N % 32 == 0 ? 2 : 0;
}
}  // namespace
}  // namespace narrow

bool qmm_narrow_covers(const void* scales, const void* biases, int K, int N, int group_size, bool silu_mul) {
  // The gated activation of a verify block is a chained launch where that has the form for it, and the chain's sums are the
  // streaming kernel's: fewer rows of such a matrix go there too, so that a token decoded alone has the bits it has in a block
  // (one row, N of both: 1024 x 4096 6.3 us there, 3.5 here; 2048 x 8192 7.4 and 6.8).
  const bool chained = silu_mul && group_size == 64 && K % 1024 == 0 && N % 128 == 0;
  // a chunk's scales of a row are one load, of 2, 4 or 8 bytes
  return !chained && narrow::tiles_for(K, N, group_size) != 0 && (((uintptr_t)scales | (uintptr_t)biases) % (256 / group_size)) == 0 &&
         (!silu_mul || N % 32 == 0);
}

int qmm_narrow_launch(const void* x, const void* w, const void* scales, const void* biases, void* y, int M, int K, int N, int group_size,
                      int act_dtype, int sb_dtype, bool silu_mul, bool packed, hipStream_t stream) {
  using namespace narrow;
  Args p{(const uint16_t*)x, w, scales, biases, (uint16_t*)y, M, K, N};
  const int tiles = tiles_for(K, N, group_size);
  const bool a16 = act_dtype == DFLASH_FP16, s16 = sb_dtype == DFLASH_FP16;
  const void* fn = tiles == 1 ? kernel_for<1>(a16, s16, group_size, silu_mul, packed) : kernel_for<2>(a16, s16, group_size, silu_mul, packed);
  constexpr int kMostLds = 16 * (2 * 4864 + 16);  // 16 rows of x
  // the attribute belongs to the device's copy of the kernel: once per device and kernel
  static bool attr_set[kMaxDevices][128] = {};
  const int idx = (((group_size >> 6) * 2 + (tiles - 1)) * 4 + (a16 ? 2 : 0) + (s16 ? 1 : 0)) * 3 + (packed ? 2 : silu_mul ? 1 : 0);
  const int slot = current_device_slot();
  if (!attr_set[slot][idx] || slot == kMaxDevices - 1) {
    DFLASH_HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kMostLds));
    attr_set[slot][idx] = true;
  }
  const int x_lds = M * (2 * K + 16), sums = kWaves * tiles * 1024;
  void* args[] = {&p};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)(N / (16 * tiles))), dim3(64 * kWaves), args, x_lds > sums ? x_lds : sums, stream));
  return DFLASH_OK;
}
}  // namespace dflash
