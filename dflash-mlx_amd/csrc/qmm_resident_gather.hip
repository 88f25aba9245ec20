// Routed experts with x in registers, for gfx950: y[p, :] = x[p, :] dequant(W[expert_ids[p]])[N, K]^T, groups of 64.
//
// The rows of an expert, 16 at a time, are an entry (build_tables() in qmm_stream_device.h); the work is all entries' tiles of 16 rows of W back
// to back, and weights of experts without rows are never touched.  A wave streams its part of K of a tile through LDS of its own, as in
// qmm_resident.h, against x of the entry in its registers; kw waves share a tile, so that each has two to five chunks of 128 k whatever K is, and
// 8 / kw such sets go through even contiguous parts of the tiles.  Sets whose part crosses into another entry fetch its rows of x there, with their
// stream drained: most do not (128 rows on 102 of 256 experts: one set in five for 2048 x 1024).  With one wave to a
// tile sums never leave it; else those of four tiles meet in LDS.  A row's sums are cut by K alone, never by what shares the call.
// us, streaming kernel -> here: 128 rows on 102 of 256 experts of 2048 x 1024 33.5 -> 28.7, of 512 x 2048 24.2 -> 19.1; 8 rows on 8 experts 10.3 -> 8.6;
// 688 rows on 128 of 1024 x 2048 42.8 -> 35.9; 512 rows on 8 of 2048 x 3072 36 -> 33.  What is left over the weights at 5.5 - 6 TB/s is 8 us of a launch: ids,
// tables, the first weights and x are a chain of trips to memory.
#include "qmm_resident.h"

namespace dflash {

int qmm_stream_grid();

namespace resident {
namespace {

struct GatherArgs {
  const uint16_t* x;  // [P, K]
  const int32_t* expert_ids;
  const char* w;  // [E, N, K/8] words
  const char* scales;
  const char* biases;
  uint16_t* y;  // [P, N]
  int P, K, N, E, kw;
  stream::Tables tab;
};

template <int NCH>
struct GatherGeometry : Geometry<64, NCH, 1> {
  static constexpr int kTables = Geometry<64, NCH, 1>::kLds;
};

template <bool H16, int NCH>
__device__ __forceinline__ void gathered_product(const GatherArgs& p) {
  using A = Act<H16>;
  using C4 = Codes<H16, 64, NCH>;
  using L = GatherGeometry<NCH>;
  constexpr int G = 2, NS = L::NS, NB = L::NB, kSlots = L::kSlots;
  extern __shared__ __align__(16) char lds[];  // every wave's ring; the waves' sums; the tables
  const int entries = stream::build_tables<64 * kWaves>(lds + L::kTables, p.tab, p.expert_ids, p.P, p.E, p.y, p.N);
  const int lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, N = p.N, tiles = N / 16, units = entries * tiles;
  const int kw = p.kw, sets = kWaves / kw, set = wave / kw, part = wave - set * kw;
  const int chunks = K / kChunk, first = part * chunks / kw, mine = (part + 1) * chunks / kw - first;
  // the set's part of the units; all sets of the workgroup make the steps of the longest
  const int all_sets = sets * (int)gridDim.x, of = set * (int)gridDim.x + (int)blockIdx.x;
  const int each_set = units / all_sets, more = units - each_set * all_sets;
  const int u0 = of * each_set + (of < more ? of : more), own = each_set + (of < more ? 1 : 0), steps = each_set + (more > 0 ? 1 : 0);
  if (steps == 0) return;

  const uint32_t w_bytes = (uint32_t)N * (uint32_t)(K / 2), s_bytes = (uint32_t)N * (uint32_t)(K / 64) * 2u;
  const auto x_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x), 0, (uint32_t)p.P * (uint32_t)K * 2u, 0x00027000);
  const uint32_t lds0 = stream::lds_address(lds), tab0 = lds0 + L::kTables;
  auto entry_word = [&](int entry) __attribute__((always_inline)) {  // rows << 16 | expert
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)stream::lds_read_u32(tab0 + p.tab.entry + 4 * entry));
  };

  // where the lanes of a load read, as in qmm_resident.h
  auto flip = [](int row) { return NCH % 4 == 0 ? row & 3 : NCH % 2 == 0 ? (row >> 1) & 1 : 0; };
  uint32_t w_at[NCH], s_at[NS];
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int granule = 64 * j + lane, row = granule / (4 * NCH), pos = granule % (4 * NCH);
    int c = (pos >> 2) ^ flip(row);
    const int piece = (pos & 3) ^ (row >> 2);
    c = first + (c < mine ? c : mine - 1);
    w_at[j] = (uint32_t)row * (uint32_t)(K / 2) + 64u * c + 16u * piece;
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int word = 4 * j + (lane & 3);
    s_at[j] = (uint32_t)(lane >> 2) * (uint32_t)(K / 32) + 4u * (first + (word < mine ? word : mine - 1));
  }
  char* const ring = lds + wave * (kDepth * L::kStage);
  struct Place {
    int entry, tile;
  };
  auto after = [&](Place at, int n) __attribute__((always_inline)) {
    at.tile += n;
    while (at.tile >= tiles) at.tile -= tiles, ++at.entry;
    return at;
  };
  auto load = [&](Place of, int d) __attribute__((always_inline)) {
    const int entry = of.entry, tile = of.tile;
    const size_t expert = entry_word(entry) & 0xFFFFu;
    const auto w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.w + expert * w_bytes), 0, w_bytes, 0x00027000);
    const auto s_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.scales + expert * s_bytes), 0, s_bytes, 0x00027000);
    const auto b_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.biases + expert * s_bytes), 0, s_bytes, 0x00027000);
    const uint32_t w_tile = (uint32_t)tile * 16u * (uint32_t)(K / 2), s_tile = (uint32_t)tile * 16u * (uint32_t)(K / 32);
    char* const at = ring + d * L::kStage;
#pragma unroll
    for (int j = 0; j < NCH; ++j) __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buf, (lds_void_t*)(at + 1024 * j), 16, w_at[j], w_tile, 0, 2);
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(s_buf, (lds_void_t*)(at + 1024 * NCH + 512 * j), 4, s_at[j], s_tile, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_buf, (lds_void_t*)(at + 1024 * NCH + 512 * j + 256), 4, s_at[j], s_tile, 0, 0);
    }
  };

  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  uint4 x[NCH][4];
  float xs[NB];
  f32x4_t from[NCH][G];
  // x of an entry, in the order of the products (rows past the entry's and chunks past `mine` are zeros), and its sums: asked for, and taken
  u32x4_t t[NCH][4];
  auto ask = [&](int entry) __attribute__((always_inline)) {
    const int rows = (int)(entry_word(entry) >> 16);
    const uint32_t row = stream::lds_read_u16(tab0 + p.tab.rows + 2 * (entry * 16 + li));
    const uint32_t x_at = (li < rows ? row * (uint32_t)K * 2u : kPast) + 256u * (uint32_t)first + 32u * q;
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        t[c][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(x_buf, (c < mine ? x_at + 256u * c + 128u * (i >> 1) + 16u * (i & 1) : kPast), 0, 0));
  };
  auto take = [&] __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) x[c][i] = stream::as_uint4(stream::permute_x(t[c][i]));
    sums_of_groups<H16, 64, NCH>(x, li, q, xs, from);
  };

  uint32_t mask = C4::kMask, magic = C4::kMagic, upper = q & 2 ? ~0u : 0u;
  asm("" : "+s"(mask), "+v"(magic), "+v"(upper));
  const uint32_t half = q & 1 ? 0u : 16u;
  auto low = [](uint32_t v) { return H16 ? f16_bits_to_f32(v & 0xFFFFu) : __uint_as_float(v << 16); };
  auto high = [](uint32_t v) { return H16 ? f16_bits_to_f32(v >> 16) : __uint_as_float(v & 0xFFFF0000u); };
  auto of_q = [&](uint32_t lo, uint32_t hi) {
    const uint32_t v = (upper & hi) | (~upper & lo);
    return H16 ? f16_bits_to_f32((v >> (16 - half)) & 0xFFFFu) : __uint_as_float((v << half) & 0xFFFF0000u);
  };
  constexpr int CX = NCH % 4 == 0 ? 4 : NCH % 2 == 0 ? 2 : 1;
  const uint32_t ring_at = lds0 + wave * (kDepth * L::kStage);
  uint32_t codes_at[CX][G];
#pragma unroll
  for (int c = 0; c < CX; ++c)
#pragma unroll
    for (int g = 0; g < G; ++g)
      codes_at[c][g] = ring_at + (uint32_t)(64 * NCH * li + 64 * (c ^ flip(li))) + 16u * ((2 * g + (q >> 1)) ^ (li >> 2)) + 8u * (q & 1);
  const uint32_t scales_at = ring_at + 1024 * NCH + 16 * li;
  const uint32_t sums_at = lds0 + L::kSums + wave * L::kSumsOfWave;

  auto emit = [&](Place of, f32x4_t sum) __attribute__((always_inline)) {
    const int entry = of.entry, tile = of.tile;
    const int rows = (int)(entry_word(entry) >> 16);
    const u32x2_t rr = stream::lds_read_u64(tab0 + p.tab.rows + 2 * (entry * 16 + 4 * q));
    const uint32_t row[4] = {rr.x & 0xFFFFu, rr.x >> 16, rr.y & 0xFFFFu, rr.y >> 16};
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * q + r < rows) p.y[(size_t)row[r] * N + 16 * tile + li] = (uint16_t)A::from_f32(sum[r]);
  };
  int held = 0;
  Place now = {u0 / tiles, 0}, met = now;  // of the step, of the first one since the last meeting
  now.tile = u0 - now.entry * tiles;
  met = now;
  // step i of the set: its unit u0 + i, at `now`
  auto step = [&](auto stage, int i) __attribute__((always_inline)) {
    constexpr int D = decltype(stage)::value;
    if (i >= own) return;
    if (now.entry != held) {
      held = now.entry;
      ask(held);
      take();
    }
    if (own - i > 1) wait_loads<L::kLoads>();
    else wait_loads<0>();
    u32x2_t w[NCH][G];
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
    if (own - i > kDepth) load(after(now, kDepth), D);
    __builtin_amdgcn_sched_barrier(0);
    f32x4_t acc = zero;
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const float sv = of_q(s[n >> 1][2 * (n & 1)], s[n >> 1][2 * (n & 1) + 1]);
      const float bv = of_q(b[n >> 1][2 * (n & 1)], b[n >> 1][2 * (n & 1) + 1]);
      acc = mfma4(xs[n], bias_of<C4>(sv, bv), acc);
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int g = 0; g < G; ++g) {
        f32x4_t d = A::mfma(x[c][2 * g], C4::unpack(w[c][g][0], mask, magic), from[c][g]);
        d = A::mfma(x[c][2 * g + 1], C4::unpack(w[c][g][1], mask, magic), d);
        const float sv = g ? high(s[c >> 2][c & 3]) : low(s[c >> 2][c & 3]);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf(sv, d[r], acc[r]);
      }
    if (kw == 1) emit(now, acc);
    else lds_write16(sums_at + 1024u * (i % kSlots) + 16u * lane, acc);
    now = after(now, 1);
  };
  // The sums of steps i0 .. i0 + 3: a set's waves deal them out
  auto meet = [&](int i0, bool more) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int n = part; n < kSlots && i0 + n < own; n += kw) {
      f32x4_t sum = zero;
      for (int v = 0; v < kw; v += 2) {
        u32x4_t f[2];
        const uint32_t at = lds0 + L::kSums + (set * kw + v) * L::kSumsOfWave + 1024u * n + 16u * lane;
        lds_read<0>(at, f[0]);
        lds_read<L::kSumsOfWave>(at, f[1]);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1])::"memory");
        const f32x4_t f0 = __builtin_bit_cast(f32x4_t, f[0]), f1 = __builtin_bit_cast(f32x4_t, f[1]);
        sum = v == 0 ? f0 + f1 : sum + f0 + f1;
      }
      emit(after(met, n), sum);
    }
    met = now;
    if (more) asm volatile("s_barrier" ::: "memory");
  };

  // x first: from the weights on, a request waits for theirs.  (A set without units reads the first one's, one with a single unit that twice.)
  const Place start = own > 0 ? now : Place{0, 0};
  held = start.entry;
  ask(held);
  __builtin_amdgcn_sched_barrier(0);
  load(start, 0);
  load(own > 1 ? after(start, 1) : start, 1);
  __builtin_amdgcn_sched_barrier(0);
  take();
  for (int i = 0; i < steps; i += kDepth) {
    step(std::integral_constant<int, 0>{}, i);
    step(std::integral_constant<int, 1>{}, i + 1);
    if (kw > 1 && (i % kSlots == kSlots - kDepth || i + kDepth >= steps)) meet(i / kSlots * kSlots, i + kDepth < steps);
  }
}

template <bool H16, int NCH>
__global__ __launch_bounds__(64 * kWaves, 2) void qmm_resident_gather_kernel(GatherArgs p) {
  gathered_product<H16, NCH>(p);
}

template <bool H16>
Kernel gather_kernel(int chunks) {
  switch (chunks) {
    case 2: return {(const void*)qmm_resident_gather_kernel<H16, 2>, GatherGeometry<2>::kTables};
    case 3: return {(const void*)qmm_resident_gather_kernel<H16, 3>, GatherGeometry<3>::kTables};
    case 4: return {(const void*)qmm_resident_gather_kernel<H16, 4>, GatherGeometry<4>::kTables};
    case 5: return {(const void*)qmm_resident_gather_kernel<H16, 5>, GatherGeometry<5>::kTables};
    default: return {nullptr, 0};
  }
}
// Waves to a tile: as few as leave each up to five chunks (six and the tables do not fit the LDS).
int waves_of_tile(int K) {
  const int chunks = K / kChunk;
  for (int kw = 1; kw <= kWaves; kw *= 2)
    if (chunks <= 5 * kw) return chunks < kw ? 0 : kw;
  return 0;
}
int chunks_of_wave(int K, int kw) {
  const int chunks = (K / kChunk + kw - 1) / kw;
  return chunks < 2 ? 2 : chunks;
}
}  // namespace
}  // namespace resident

// expert_ids on the device; P rows, E experts within the tables' limits (the caller has asked the streaming kernel's rule).  Beyond K = 4096 every wave
// has four and a half to five chunks of each tile, and where experts have four rows and more the streaming kernel is as fast or faster (us there and here:
// 32 rows on 8 experts of 5120 x 4096 20.6 / 22.8, 128 rows 31.9 / 34.3; 128 rows on 8 of 5120 x 2048 20.2 / 23.8, on 16 of 4608 x 2048 20.4 / 23.6, 256 on 32
// of 4608 x 1024 20.8 / 23.9; with fewer 8 rows on 8 of 5120 x 4096 18.9 / 18.7, 2 rows 11.3 / 9.4, 32 on 256 of 4608 x 1024 as fast).  Up to there it is
// slower only where 128 - 256 rows meet on 1000 - 1600 tiles (128 on 8 of 2560 x 2048 14.0 / 15.8, of 3584 x 2048 16.4 / 18.0), else 5 - 30 % faster.
bool qmm_resident_gather_covers(const void* scales, const void* biases, int P, int K, int N, int E, int group_size, int act_dtype, int sb_dtype) {
  using namespace resident;
  if (group_size != 64 || act_dtype != sb_dtype || K % kChunk != 0 || N % 16 != 0 || (((uintptr_t)scales | (uintptr_t)biases) % 4) != 0) return false;
  if (K > 4096 && N > 512 && P >= 4 * E) return false;
  const int kw = waves_of_tile(K);
  if (kw == 0 || (long long)N * K / 2 >= (1ll << 31) || (long long)P * K * 2 >= (1ll << 31)) return false;
  const int most = stream::most_entries(P, E);
  const Kernel k = gather_kernel<false>(chunks_of_wave(K, kw));
  return (long long)most * (N / 16) < (1ll << 30) && k.fn != nullptr && k.lds + stream::Tables(E, most).bytes <= 160 * 1024;
}

int qmm_resident_gather_launch(const void* x, const int32_t* expert_ids, const void* w, const void* scales, const void* biases, void* y, int P,
                               int K, int N, int E, int dtype, hipStream_t stream) {
  using namespace resident;
  const bool h16 = dtype == DFLASH_FP16;
  const int kw = waves_of_tile(K), chunks = chunks_of_wave(K, kw);
  const Kernel k = h16 ? gather_kernel<true>(chunks) : gather_kernel<false>(chunks);
  GatherArgs p{(const uint16_t*)x, expert_ids, (const char*)w, (const char*)scales, (const char*)biases, (uint16_t*)y, P, K, N, E, kw,
               stream::Tables(E, stream::most_entries(P, E))};
  static bool attr_set[kMaxDevices][2][8] = {};
  const int slot = current_device_slot();
  bool& done = attr_set[slot][h16][chunks];
  if (!done || slot == kMaxDevices - 1) {
    DFLASH_HIP_OK(hipFuncSetAttribute(k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    done = true;
  }
  void* args[] = {&p};
  DFLASH_HIP_OK(hipLaunchKernel(k.fn, dim3((unsigned)qmm_stream_grid()), dim3(64 * kWaves), args, k.lds + p.tab.bytes, stream));
  return DFLASH_OK;
}
}  // namespace dflash
