// 4-bit affine matmul for any number of rows, y[M,N] = x[M,K] . round(s*q + b)^T (gfx950): prompts,
// and every other call the 16-row kernels do not serve.
//
// What the reference leaves to mx.quantized_matmul (dflash_mlx/verify_qmm.py:277-280).  A weight is
// dequantised to the activation type as the array-op form of this package does it (s*q + b in
// fp32, rounded once) and multiplied on the matrix cores with fp32 accumulation.
//
// The contraction is bound by the matrix cores from about 100 rows on and by the weights' 0.56 B
// below that; what it must not pay for is dequantising a weight more often than once per block
// of rows.  So a wave owns whole columns: a workgroup is 4 waves side by side, each 16*NT columns
// wide and all 16*MT rows high, weights go from memory straight to registers (a lane's 16 bytes
// are 32 consecutive k of one row, exactly one scale and bias for every group size) and only x,
// which all four waves read, goes through LDS, double-buffered.  k is fed to the matrix core in the
// order the packed words have it: step j of an iteration multiplies word j of every lane, and x is
// read from LDS in that order.
//
//  * dequantisation: code q sits in the low bits of a half word; as an fp16 subnormal that half is
//    q 2^-24, so fma_mix(half, s 2^24, b) is s q + b in one instruction and exact up to its one
//    rounding; the conversion to the activation type packs two at a time: 19 vector instructions per
//    8 weights.
//  * W is the A operand (rows of the tile = columns of y), x the B operand, and the columns of a
//    wave are dealt to its tiles so that a lane ends up with 4*NT consecutive columns of one row.
//  * The (tile, k) space is divided evenly among a grid that fills the chip once: a workgroup
//    whose range covers all of K for a tile writes y, the others leave fp32 partial tiles in the
//    workspace, and whoever arrives last at a tile adds them in order of k.  Nobody waits.
//    Deterministic.  Calls with many more tiles than workgroups take one tile per workgroup.
#include "dflash_common.h"
#include "qmm_stream_device.h"

namespace dflash {
namespace rows {

constexpr int kThreads = 256;
constexpr int kWaves = 4;

struct Args {
  const uint16_t* x;
  const uint32_t* w;
  const uint16_t* scales;
  const uint16_t* biases;
  uint16_t* y;
  float* partials;      // [2 * grid][tile of 16x16 in the workgroup][thread][4]
  uint32_t* counters;   // one per tile, zero between calls
  int M, K, N;
  int group_shift;      // log2(group size / 32)
  int sb_fp16;
  int tiles_m, tiles, iters;  // iters = ceil(K / k per iteration)
  int split;            // 0: one tile per workgroup
};

typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;

template <bool FP16>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (FP16) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{a, b}), f16x2_t));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{a, b}), bf16x2_t));
  }
}
__device__ __forceinline__ float code_fma(uint32_t pair, int hi, float s24, float b) {
  const f16x2_t h = __builtin_bit_cast(f16x2_t, pair);
  return __builtin_fmaf((float)h[hi], s24, b);
}
// eight codes of one word (k ascending from the low nibble) -> eight values of the activation type
template <bool FP16>
__device__ __forceinline__ uint4 dequant8(uint32_t w, float s24, float b, uint32_t mask) {
  const uint32_t p0 = w & mask, p1 = (w >> 4) & mask, p2 = (w >> 8) & mask, p3 = (w >> 12) & mask;  // (k0,k4) (k1,k5) ..
  uint4 r;
  r.x = pack2<FP16>(code_fma(p0, 0, s24, b), code_fma(p1, 0, s24, b));
  r.y = pack2<FP16>(code_fma(p2, 0, s24, b), code_fma(p3, 0, s24, b));
  r.z = pack2<FP16>(code_fma(p0, 1, s24, b), code_fma(p1, 1, s24, b));
  r.w = pack2<FP16>(code_fma(p2, 1, s24, b), code_fma(p3, 1, s24, b));
  return r;
}
__device__ __forceinline__ float sb_value(uint32_t h, int fp16) {
  return fp16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
}

// WPL: packed words of a row that a lane holds per iteration; an iteration is 32 WPL k.
template <bool FP16, int MT, int NT, int WPL>
__global__ __launch_bounds__(kThreads, MT * NT > 12 ? 2 : 3) void qmm_rows_kernel(Args a) {
  using A = stream::Act<FP16>;
  constexpr int BM = 16 * MT, BN = kWaves * 16 * NT;
  constexpr int kStepK = 32 * WPL;
  constexpr int kGran = kStepK / 8;             // 16-byte granules of an x row and iteration
  constexpr int kXRows = kThreads / kGran;      // rows of x that the workgroup loads at a time
  constexpr int XL = (BM + kXRows - 1) / kXRows;
  constexpr int kStageBytes = BM * kStepK * 2;
  extern __shared__ __attribute__((aligned(1024))) char lds[];  // 2 stages of x
  __shared__ uint32_t s_last;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kblk = lane >> 4;
  const int grid = (int)gridDim.x;
  // neighbours in tile order (same columns, other rows) behind one L2
  const int wg = grid % 8 == 0 ? (int)(blockIdx.x % 8) * (grid / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  long long u, u1;
  if (a.split) {
    const long long units = (long long)a.tiles * a.iters;
    u = units * wg / grid;
    u1 = units * (wg + 1) / grid;
  } else {
    u = (long long)wg * a.iters;
    u1 = u + a.iters;
  }
  const int first_tile = (int)(u / a.iters);
  const int G = a.K >> (5 + a.group_shift);
  uint32_t mask = 0x000F000Fu;
  asm volatile("" : "+s"(mask));

  // this thread's part of an x stage: granule tid % kGran of rows tid / kGran + kXRows i
  const int xg = tid % kGran, xr = tid / kGran;

  while (u < u1) {
    const int tile = (int)(u / a.iters);
    const int it0 = (int)(u - (long long)tile * a.iters);
    const long long tile_end = (long long)(tile + 1) * a.iters;
    const int it1 = (int)((u1 < tile_end ? u1 : tile_end) - (long long)tile * a.iters);
    const int nb = tile / a.tiles_m, mb = tile - nb * a.tiles_m;
    const int m0 = mb * BM, n0 = nb * BN + wave * 16 * NT;
    const int nsafe = n0 < a.N ? n0 : 0;  // (a wave past the last column reads the first rows and stores nothing)

    // uniform bases of this tile and 32-bit byte offsets of this lane's rows from them
    const char* xbase = (const char*)(a.x + (size_t)m0 * a.K);
    const char* wbase = (const char*)a.w + (size_t)nsafe * (a.K >> 1);
    const char* sbase = (const char*)(a.scales + (size_t)nsafe * G);
    const char* bbase = (const char*)(a.biases + (size_t)nsafe * G);
    uint32_t xo[XL], wo[NT], so[NT];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      int row = xr + kXRows * i;
      row = m0 + row < a.M ? row : a.M - 1 - m0;
      xo[i] = (uint32_t)row * (uint32_t)a.K * 2u + xg * 16;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      int row = 4 * NT * (li >> 2) + 4 * t + (li & 3);
      row = nsafe + row < a.N ? row : a.N - 1 - nsafe;
      wo[t] = (uint32_t)(row * (a.K >> 1));
      so[t] = (uint32_t)(row * G * 2);
    }
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    uint4 xv[XL];          // x stage on its way to LDS
    uint32_t wn[NT][WPL];  // codes, scales, biases of the next iteration
    uint32_t sn[NT], bn[NT];
    auto load_x = [&](int it) __attribute__((always_inline)) {
      const bool in = it * kStepK + xg * 8 < a.K;  // granules past K are zero
#pragma unroll
      for (int i = 0; i < XL; ++i) {
        xv[i] = *reinterpret_cast<const uint4*>(xbase + (xo[i] + (in ? (uint32_t)it * (kStepK * 2) : 0u - xg * 16)));
        if (!in) xv[i] = make_uint4(0u, 0u, 0u, 0u);
      }
    };
    auto load_w = [&](int it) __attribute__((always_inline)) {
      const int k = it * kStepK + kblk * (8 * WPL);
      const bool in = k < a.K;
      const int g = in ? (k >> 5) >> a.group_shift : 0;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const char* src = wbase + (wo[t] + (in ? (uint32_t)k >> 1 : 0u));
        if constexpr (WPL == 4) {
          const uint4 v = *reinterpret_cast<const uint4*>(src);
          wn[t][0] = v.x, wn[t][1] = v.y, wn[t][2] = v.z, wn[t][3] = v.w;
        } else {
          const uint2 v = *reinterpret_cast<const uint2*>(src);
          wn[t][0] = v.x, wn[t][1] = v.y;
        }
        sn[t] = *reinterpret_cast<const uint16_t*>(sbase + (so[t] + (uint32_t)g * 2));
        bn[t] = *reinterpret_cast<const uint16_t*>(bbase + (so[t] + (uint32_t)g * 2));
        if (!in) sn[t] = bn[t] = 0u;  // weights past K are zero
      }
    };
    auto store_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < XL; ++i) {
        const int row = xr + kXRows * i;
        if (BM % kXRows == 0 || row < BM)
          *reinterpret_cast<uint4*>(lds + buf * kStageBytes + row * (kGran * 16) + ((xg ^ (row & 7)) << 4)) = xv[i];
      }
    };

    load_x(it0);
    load_w(it0);
    store_x(0);
    if (it0 + 1 < it1) load_x(it0 + 1);
    __syncthreads();
    for (int it = it0; it < it1; ++it) {
      const int buf = (it - it0) & 1;
      uint32_t wc[NT][WPL];
      float sc[NT], bc[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int j = 0; j < WPL; ++j) wc[t][j] = wn[t][j];
        sc[t] = sb_value(sn[t], a.sb_fp16) * 16777216.0f;
        bc[t] = sb_value(bn[t], a.sb_fp16);
      }
      if (it + 1 < it1) {
        store_x(buf ^ 1);
        load_w(it + 1);
        if (it + 2 < it1) load_x(it + 2);
      }
      const char* xs = lds + buf * kStageBytes;
#pragma unroll
      for (int j = 0; j < WPL; ++j) {
        uint4 wf[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          wf[t] = dequant8<FP16>(wc[t][j], sc[t], bc[t], mask);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const uint4 xf = *reinterpret_cast<const uint4*>(xs + (16 * i + li) * (kGran * 16) + (((WPL * kblk + j) ^ (li & 7)) << 4));
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[i][t] = A::mfma(wf[t], xf, acc[i][t]);
        }
      }
      __syncthreads();
    }

    const bool whole = it0 == 0 && it1 == a.iters;
    // accumulator r of lane (li, kblk), tile (i, t): row m0 + 16 i + li, column n0 + 4 NT kblk + 4 t + r
    auto emit = [&](int i, const f32x4_t (&v)[NT]) __attribute__((always_inline)) {
      const int m = m0 + 16 * i + li, n = n0 + 4 * NT * kblk;
      if (m >= a.M) return;
      uint16_t* dst = a.y + (size_t)m * a.N + n;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint2 o = make_uint2(pack2<FP16>(v[t][0], v[t][1]), pack2<FP16>(v[t][2], v[t][3]));
        if (n + 4 * t < a.N) *reinterpret_cast<uint2*>(dst + 4 * t) = o;
      }
    };
    if (whole) {
#pragma unroll
      for (int i = 0; i < MT; ++i) emit(i, acc[i]);
    } else {
      // slot 0 of a workgroup: the tile its range starts in, slot 1: the one it ends in
      const int which = tile == first_tile ? 0 : 1;
      constexpr size_t kSlotFloats = (size_t)BM * BN;
      auto slot = [&](int w, int s) __attribute__((always_inline)) { return a.partials + ((size_t)w * 2 + s) * kSlotFloats; };
      float* mine = slot(wg, which) + tid * 4;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) stream::store_partial(mine + (i * NT + t) * (kThreads * 4), acc[i][t]);
      // every wave's stores are acknowledged before the arrival is counted
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      const long long units = (long long)a.tiles * a.iters, lo = (long long)tile * a.iters, hi = lo + a.iters;
      // the workgroup that holds unit v: ceil((v + 1) * grid / units) - 1
      const int lo_wg = (int)(((lo + 1) * grid + units - 1) / units) - 1;
      const int hi_wg = (int)((hi * grid + units - 1) / units) - 1;
      if (tid == 0) s_last = atomicInc(&a.counters[tile], (uint32_t)(hi_wg - lo_wg)) == (uint32_t)(hi_wg - lo_wg);
      __syncthreads();
      if (s_last) {
        // only the first contributor can have started before the tile (then it ends in it)
        const int which_first = units * lo_wg / grid < lo ? 1 : 0;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          f32x4_t sum[NT];
#pragma unroll
          for (int t = 0; t < NT; ++t) sum[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          for (int c = lo_wg; c <= hi_wg; ++c) {
            if (c == wg) {
#pragma unroll
              for (int t = 0; t < NT; ++t) sum[t] += acc[i][t];
            } else {
              const float* src = slot(c, c == lo_wg ? which_first : 0) + (size_t)i * NT * (kThreads * 4) + tid * 4;
#pragma unroll
              for (int t = 0; t < NT; ++t) {
                f32x4_t v;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  v[r] = __hip_atomic_load(src + t * (kThreads * 4) + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sum[t] += v;
              }
            }
          }
          emit(i, sum);
        }
      }
      __syncthreads();
    }
    u += it1 - it0;
  }
}

// Registers decide: the large tiles keep 64 k in flight, the others 128.
constexpr int words_per_lane(int mt, int nt) { return mt * nt > 16 ? 2 : 4; }

template <bool FP16>
const void* kernel_for(int mt, int nt) {
#define DFLASH_ROWS_PICK(MT, NT) \
  if (mt == MT && nt == NT) return (const void*)qmm_rows_kernel<FP16, MT, NT, words_per_lane(MT, NT)>;
  DFLASH_ROWS_PICK(1, 2) DFLASH_ROWS_PICK(2, 2) DFLASH_ROWS_PICK(3, 2) DFLASH_ROWS_PICK(4, 2) DFLASH_ROWS_PICK(5, 2)
  DFLASH_ROWS_PICK(6, 2) DFLASH_ROWS_PICK(8, 2)
  DFLASH_ROWS_PICK(4, 4) DFLASH_ROWS_PICK(5, 4) DFLASH_ROWS_PICK(6, 4) DFLASH_ROWS_PICK(8, 4)
#undef DFLASH_ROWS_PICK
  return nullptr;
}

struct Plan {
  int mt, nt, tiles_m, tiles, iters, grid, split;
  size_t workspace;
};

constexpr size_t kCounterBytes = 64 * 1024;

bool covers(int M, int K, int N, int group_size) {
  return M > 0 && K > 0 && N > 0 && (group_size == 32 || group_size == 64 || group_size == 128) && K % group_size == 0 &&
         N % 16 == 0;
}

Plan plan(int M, int K, int N, int cus) {
  Plan p;
  // rows: as few blocks of at most 128 as cover M, each no higher than it has to be
  p.tiles_m = (M + 127) / 128;
  const int per = (M + p.tiles_m - 1) / p.tiles_m;
  p.mt = (per + 15) / 16;
  if (p.mt == 7) p.mt = 8;
  p.tiles_m = (M + 16 * p.mt - 1) / (16 * p.mt);
  p.nt = p.mt >= 6 ? 4 : 2;
  const int bn = kWaves * 16 * p.nt;
  p.tiles = p.tiles_m * ((N + bn - 1) / bn);
  const int step = 32 * words_per_lane(p.mt, p.nt);
  p.iters = (K + step - 1) / step;
  const int slots = cus * (p.mt * p.nt > 12 ? 2 : 3);
  const long long units = (long long)p.tiles * p.iters;
  if (p.tiles >= 8 * slots || p.tiles > (int)(kCounterBytes / 4)) {
    p.split = 0;
    p.grid = p.tiles;
    p.workspace = 0;
  } else {
    p.split = 1;
    p.grid = units < slots ? (int)units : slots;
    p.workspace = kCounterBytes + (size_t)p.grid * 2 * (16 * p.mt) * bn * sizeof(float);
  }
  return p;
}

}  // namespace rows

int qmm_stream_grid();
}  // namespace dflash

extern "C" size_t dflash_qmm_rows_workspace_bytes(int M, int K, int N, int group_size) {
  using namespace dflash;
  if (!rows::covers(M, K, N, group_size)) return 0;
  return rows::plan(M, K, N, qmm_stream_grid()).workspace;
}

extern "C" int dflash_qmm_rows(const void* x, const uint32_t* w_q, const void* scales, const void* biases, void* y,
                               void* workspace, size_t workspace_bytes, int M, int K, int N, int group_size,
                               int act_dtype, int sb_dtype, void* stream) {
  using namespace dflash;
  DFLASH_REQUIRE(x && w_q && scales && biases && y, DFLASH_ERR_ARG, "dflash_qmm_rows: null operand");
  DFLASH_REQUIRE((act_dtype == DFLASH_BF16 || act_dtype == DFLASH_FP16) && (sb_dtype == DFLASH_BF16 || sb_dtype == DFLASH_FP16),
                 DFLASH_ERR_ARG, "dflash_qmm_rows: activations and scales must be bf16/fp16");
  DFLASH_REQUIRE(rows::covers(M, K, N, group_size), DFLASH_ERR_SHAPE,
                 "dflash_qmm_rows: need M > 0, group_size in {32,64,128}, K %% group_size == 0, N %% 16 == 0 (M=%d K=%d N=%d gs=%d)",
                 M, K, N, group_size);
  DFLASH_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)w_q % 16) == 0 && ((uintptr_t)y % 8) == 0, DFLASH_ERR_ARG,
                 "dflash_qmm_rows: x and w_q must be 16-byte aligned");
  const rows::Plan p = rows::plan(M, K, N, qmm_stream_grid());
  DFLASH_REQUIRE(p.workspace == 0 || (workspace && workspace_bytes >= p.workspace), DFLASH_ERR_WORKSPACE,
                 "dflash_qmm_rows: workspace of %zu bytes needed, %zu given", p.workspace, workspace ? workspace_bytes : (size_t)0);
  rows::Args a;
  a.x = (const uint16_t*)x; a.w = w_q; a.scales = (const uint16_t*)scales; a.biases = (const uint16_t*)biases;
  a.y = (uint16_t*)y;
  a.counters = (uint32_t*)workspace;
  a.partials = workspace ? (float*)((char*)workspace + rows::kCounterBytes) : nullptr;
  a.M = M; a.K = K; a.N = N;
  a.group_shift = group_size == 32 ? 0 : group_size == 64 ? 1 : 2;
  a.sb_fp16 = sb_dtype == DFLASH_FP16;
  a.tiles_m = p.tiles_m; a.tiles = p.tiles; a.iters = p.iters; a.split = p.split;
  const bool fp16 = act_dtype == DFLASH_FP16;
  const void* fn = fp16 ? rows::kernel_for<true>(p.mt, p.nt) : rows::kernel_for<false>(p.mt, p.nt);
  const int lds_bytes = 2 * 16 * p.mt * (32 * rows::words_per_lane(p.mt, p.nt)) * 2;
  static bool attr_set[kMaxDevices][2][9][5] = {};
  const int dev = current_device_slot();
  if (lds_bytes > 48 * 1024) {
    bool& set = attr_set[dev][fp16][p.mt][p.nt];
    if (!set || dev == kMaxDevices - 1) {
      DFLASH_HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes));
      set = true;
    }
  }
  void* args[] = {&a};
  DFLASH_HIP_OK(hipLaunchKernel(fn, dim3((unsigned)p.grid), dim3(rows::kThreads), args, (size_t)lds_bytes, (hipStream_t)stream));
  return DFLASH_OK;
}
