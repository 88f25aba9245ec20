// Host side of qmm_resident.h: which products of up to 16 rows its kernel takes, and how their K range is cut.
#include "qmm_resident.h"

namespace dflash {

int qmm_stream_grid();

namespace resident {
namespace {
constexpr int kRowCounters = 16384;  // the any-rows product's workspace: 64 KiB of counters (here: one per workgroup of a slice), then tiles
constexpr int kMostRowSlices = 8;

struct Plan {
  int chunks;  // NCH of the kernel, 0: not this kernel's
  int slices;
  int cus;
  size_t workspace;
  bool padded;  // qmm_narrow's where that has the shape
};
// One row of K <= 1024 against few rows of W is qmm_narrow's, which has no ring to set up (1024 x 512, 1 / 16 rows: 3.1 / 3.7 us there, 3.7 /
// 3.8 here; 1024 x 8192 5.3 / 5.9 there, 4.8 / 5.0 here), and so is a K that leaves more than a third of the waves' chunks empty: 1152 x 2048 3.5 / 4.4 there and
// 4.0 / 4.2 here, 2304 x 1024 in groups of 128 3.9 / 6.0 and 5.2 / 5.6.  With fuller waves a verify block gains what one row loses, or more (1536 x 2048
// 3.8 / 4.7 and 4.0 / 4.2, 2560 x 2048 4.5 / 6.5 and 4.6 / 4.9, 3072 x 2048 in groups of 128 4.5 / 6.8 and 5.3 / 5.6; 3072 x 2048 5.2 / 7.3 and 4.6 / 5.1).
// A row's bits must not depend on the rows beside it, so there is one kernel for both.
//
// Slices by a model fitted to 1000 calls of 1 and 16 rows with every number of them (K from 2048 to 24576, N from 1024 to 32768, all group sizes,
// weights from memory and from the cache): in 10 ns and less what all have, 80 per chunk for x and the first tile, 35 + 9 per chunk for each further tile
// of the busiest workgroup (groups of 32: 96 and 4) and 8 per chunk for each of the mean one, 110 for the meeting of slices and, for an odd number of chunks, whose runs of 64
// bytes share their lines with other waves, 1 per MB.  What it picks is within 0.3 % of the best in the mean and 6 % at most.  us for 16 rows, 1 / 2 / 3 / 4
// slices: 4096 x 5120 7.3 / 6.8 / 7.1 / 8.9; 5120 x 4096 7.6 / 7.4 / 6.8 / 7.6; 6144 x 4096 8.3 / 7.7 / 6.9 / 7.8; 12288 x 4096 - / 11.7 / 10.8 / 10.5; 14336 x 8192
// - / - / 19.9 / 18.0; 17408 x 5120 - / - / 15.9 / 16.6 (K x N).  M does not enter: a row must not change with the rows beside it.  (The tile that a few
// workgroups have more than the others counts in full: 14336 x 4096 in three slices has 256 tiles for 85 workgroups, 13.3, in four slices 11.7; the
// streaming kernel 13.0.)
//
// Where N / 128 divides the compute units, the streaming kernel (groups of 64) has equal parts without a remainder and is at its best: there the call is
// its own if a model of either says so (2.5 % rms over 71 such shapes).  us there and here: 9216 x 16384 21.2 / 22.3, 12800 x 16384 27.5 / 29.4,
// 6400 x 32768 27.4 / 28.9, 17408 x 8192 21.4 / 22.5; 16384 x 8192 19.7 / 18.3.  Waves that are a third empty and more also lose to it on wide matrices
// whose N / 128 is a multiple of the compute units (1280 x 65536 13.5 / 14.6, 1024 x 65536 in groups of 32 13.2 / 15.6, 2304 x 32768 in groups of 128
// 12.0 / 12.9), half empty ones on any but those between 32768 and 65536, where its parts are uneven (1024 x 28672 7.3 / 8.4, 1024 x 151936 25.7 / 28.8;
// 1024 x 40960 10.8 / 10.5).
Plan make_plan(int K, int N, int group_size, int cus) {
  const int step = group_size == 128 ? 2 : 1, most = most_chunks(group_size, 1);
  if ((group_size != 32 && group_size != 64 && group_size != 128) || K % (kChunk * step) != 0 || N % 16 != 0 || N < 16) return {0, 0, cus, 0, false};
  if (K <= 1024 && N <= 4096) return {0, 0, cus, 0, false};
  if ((long long)N * K / 2 >= (1ll << 31) - (1 << 24)) return {0, 0, cus, 0, false};  // 32-bit byte offsets, and kPast behind them
  const int pieces = K / (kChunk * step), tiles = N / 16;
  const double megabytes = 1e-6 * N * K * (0.5 + 4.0 / group_size), first = group_size == 32 ? 96.0 : 80.0, further = group_size == 32 ? 4.0 : 9.0;
  Plan best = {0, 0, cus, 0, false};
  double best_cost = 0.0;
  for (int slices = 1; slices <= kMostSlices; ++slices) {
    const int parts = kWaves * slices;
    if (pieces < parts || slices > cus) break;
    int chunks = step * ((pieces + parts - 1) / parts);
    if (chunks > most) continue;
    if ((long long)(slices - 1) * N > 65536) break;  // every other slice keeps a KiB per tile in the workspace that the streaming kernel asks for
    if (chunks < 2) chunks = 2;
    const int lanes = tiles < cus / slices ? tiles : cus / slices, more = (tiles + lanes - 1) / lanes - 1;
    double cost = first * chunks + more * (35.0 + further * chunks) + 8.0 * chunks * ((double)tiles / lanes - 1.0);
    if (slices > 1) cost += 110.0;
    if (chunks % 2 != 0) cost += megabytes;
    if (best.chunks == 0 || cost < best_cost) best.chunks = chunks, best.slices = slices, best_cost = cost;
  }
  if (best.slices > 1 && group_size == 64 && N % 128 == 0 && N >= 4096 && cus % (N / 128) == 0) {
    const double us = 1.83 + 0.0109 * best_cost + 0.058 * megabytes, streaming_us = 7.2 + (K % 512 == 0 ? 0.171 : 0.186) * megabytes;
    if (us > streaming_us) return {0, 0, cus, 0, false};
  }
  const bool padded = 3 * pieces * step < 2 * kWaves * best.slices * best.chunks;
  if (padded && best.slices == 1 && N > 20480 &&
      ((N % 128 == 0 && N / 128 % cus == 0) || (K <= 1024 && group_size == 64 && (N <= 32768 || N >= 65536)))) return {0, 0, cus, 0, false};
  best.padded = padded && N <= 4096;
  best.workspace = best.slices < 2 ? 0 : (size_t)64 * 1024 + (size_t)tiles * (best.slices - 1) * 1024;
  return best;
}

// The last few plans of this thread: a model asks for the same ones over and over (0.15 us each).
const Plan& plan_for(int K, int N, int group_size) {
  struct Entry {
    int K, N, group_size;
    Plan p;
  };
  static thread_local Entry cache[64] = {};
  const int cus = qmm_stream_grid();
  Entry& e = cache[((unsigned)K * 2654435761u + (unsigned)N * 40503u * 65537u + (unsigned)group_size) >> 26];
  if (e.K != K || e.N != N || e.group_size != group_size || e.p.cus != cus) e = Entry{K, N, group_size, make_plan(K, N, group_size, cus)};
  return e.p;
}
}  // namespace
}  // namespace resident

bool qmm_resident_covers(const void* scales, const void* biases, size_t workspace_bytes, int K, int N, int group_size, int act_dtype,
                         int sb_dtype, bool narrow) {
  // (mixed types: the streaming kernel's; a lane's words of scales are four bytes)
  if (act_dtype != sb_dtype || (((uintptr_t)scales | (uintptr_t)biases) % 4) != 0) return false;
  if (K <= 1024 && N <= 4096) return false;  // as in make_plan, without looking the plan up
  const resident::Plan& plan = resident::plan_for(K, N, group_size);
  return plan.chunks != 0 && !(narrow && plan.padded) && workspace_bytes >= plan.workspace;
}

int qmm_resident_launch(const void* x, const void* w, const void* scales, const void* biases, void* y, void* workspace, int M, int K,
                        int N, int group_size, int dtype, bool silu_mul, bool packed, int spin_limit, hipStream_t stream) {
  using namespace resident;
  const Plan& plan = plan_for(K, N, group_size);
  const bool h16 = dtype == DFLASH_FP16;
  const Kernel k = h16 ? fp16_kernel(group_size, plan.chunks, silu_mul, packed) : bf16_kernel(group_size, plan.chunks, silu_mul, packed);
  DFLASH_REQUIRE(k.fn != nullptr, DFLASH_ERR_SHAPE, "dflash_qmm_m16: no kernel for K=%d N=%d gs=%d", K, N, group_size);
  if (spin_limit <= 0) spin_limit = option(DFLASH_OPT_QMM_SPIN_LIMIT) > 0 ? option(DFLASH_OPT_QMM_SPIN_LIMIT) : stream::kSpinLimit;
  Args p{(const uint16_t*)x, w, scales, biases, (uint16_t*)y, (float*)((char*)workspace + 64 * 1024), (uint32_t*)workspace,
         M, K, N, plan.slices, spin_limit, 0, 0, 0, 0, 0};
  set_partition(p, group_size, plan.cus);
  // the attribute belongs to the device's copy of the kernel: once per device and kernel
  static bool attr_set[kMaxDevices][2][3][8][4] = {};
  const int slot = current_device_slot();
  bool& done = attr_set[slot][h16][group_size >> 6][plan.chunks][(silu_mul ? 1 : 0) + (packed ? 2 : 0)];
  if (!done || slot == kMaxDevices - 1) {
    DFLASH_HIP_OK(hipFuncSetAttribute(k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, k.lds));
    done = true;
  }
  void* args[] = {&p};
  DFLASH_HIP_OK(hipLaunchKernel(k.fn, dim3((unsigned)(p.slices * p.lanes)), dim3(64 * kWaves), args, k.lds, stream));
  return DFLASH_OK;
}

// Tiles of 16 rows: two at least, which is what a call of up to 16 rows takes whose K or columns the kernel for those does not serve (rows that are not
// there are read as zeros and not stored).  16 rows, us, through the any-rows product
// and here: 10496 x 352 12.1 / 7.3, 4096 x 3936 in groups of 32 10.9 / 7.9, 2688 x 2880 in groups of 32 9.8 / 6.4, 1536 x 1632 with the activation 8.7 / 5.2;
// three rows of 10752 x 320 11.2 / 7.0.
int row_tiles_of(int M) { return M <= 32 ? 2 : (M + 15) / 16; }

// Up to 80 rows: the slices of K that take the least time by a model fitted to 328 combinations of 25 matrices, 32 to 80 rows and 1 to 6
// slices (4.7 % rms, what it picks is within 3 % of the best of its call).  The caller takes this kernel where that is less than what the any-rows
// product is expected to take: 17 - 32 rows of most matrices (4096 x 4096 10.3 -> 7.5 us, 4096 x 12288 19.9 -> 12.9, 5120 x 34816 with the activation 40.7 -> 30.5),
// 33 - 48 of those too (4096 x 6144 15.1 -> 11.1; of 5120 x 34816 with the activation as long as there, 44), up to 80 of fewer (80 rows of 4096 x 6144 17.5 -> 13.8).  The others stay there (4096 x 24576
// with the activation, 80 rows: 30.8 there, 33.8 here: sums of eight waves for every 16 x 16 piece, and x of 80 rows leaves room for two chunks a wave only).
// Of 193 calls of 18 matrices what is taken is within 0.2 % of the better of the two in the mean and 4 % at most (2.5 and 33 % before the factor below).
bool qmm_resident_rows_plan(int M, int K, int N, int group_size, bool silu_mul, int* chunks_out, int* slices_out, double* us_out, size_t* workspace) {
  using namespace resident;
  const int row_tiles = row_tiles_of(M), step = group_size == 128 ? 2 : 1;
  if (M < 1 || row_tiles > kMostRowTiles || K % (kChunk * step) != 0 || N % 16 != 0 || (long long)N * K / 2 >= (1ll << 31) - (1 << 24))
    return false;
  const int pieces = K / (kChunk * step), tiles = N / 16, cus = qmm_stream_grid(), most = most_chunks(group_size, row_tiles);
  if (cus > kRowCounters) return false;
  bool found = false;
  for (int slices = 1; slices <= kMostRowSlices && slices <= cus && pieces >= kWaves * slices; ++slices) {
    const int parts = kWaves * slices, fewest = step * ((pieces + parts - 1) / parts), chunks = fewest < 2 ? 2 : fewest;
    if (chunks > most) continue;
    const int lanes = cus / slices, more_tiles = (20 * tiles + 19 * lanes - 1) / (20 * lanes) - 1;  // (of the busiest workgroup, but for a lane in 20)
    double us = 3.1 + 0.536 * row_tiles * chunks + more_tiles * (0.847 * chunks - 0.7 + (0.353 - 0.051 * chunks) * row_tiles) + (silu_mul ? 0.19 : 0.0);
    if (slices > 1) us += 0.84 + 0.25 * slices - 0.3 * row_tiles * (more_tiles + 1) + 1.12e-3 * tiles * row_tiles * slices;
    if (!found || us < *us_out) *chunks_out = chunks, *slices_out = slices, *us_out = us, found = true;
  }
  // (measured again beside the any-rows product's own model, 193 calls of 17 to 80 rows: 0.91 of that for two row tiles, 0.94 for five)
  if (found) *us_out *= 0.81 + 0.025 * row_tiles;
  if (found) *workspace = *slices_out < 2 ? 0 : (size_t)4 * kRowCounters + (size_t)tiles * row_tiles * *slices_out * 1024;
  return found;
}

// scales and biases on 4 bytes, of the activations' type
int qmm_resident_rows_launch(const void* x, const void* w, const void* scales, const void* biases, void* y, void* workspace, int M, int K,
                             int N, int group_size, int dtype, bool silu_mul, int chunks, int slices, hipStream_t stream) {
  using namespace resident;
  const int row_tiles = row_tiles_of(M);
  const bool h16 = dtype == DFLASH_FP16;
  const Kernel k = h16 ? fp16_rows_kernel(row_tiles, group_size, chunks, silu_mul) : bf16_rows_kernel(row_tiles, group_size, chunks, silu_mul);
  DFLASH_REQUIRE(k.fn != nullptr, DFLASH_ERR_SHAPE, "dflash_qmm_rows: no kernel for M=%d K=%d N=%d gs=%d", M, K, N, group_size);
  Args p{(const uint16_t*)x, w, scales, biases, (uint16_t*)y, workspace ? (float*)((char*)workspace + 4 * kRowCounters) : nullptr,
         (uint32_t*)workspace, M, K, N, slices, 0, 0, 0, 0, 0, 0};
  set_partition(p, group_size, qmm_stream_grid());
  static bool attr_set[kMaxDevices][2][3][8][kMostRowTiles + 1][2] = {};
  const int slot = current_device_slot();
  bool& done = attr_set[slot][h16][group_size >> 6][chunks][row_tiles][silu_mul];
  if (!done || slot == kMaxDevices - 1) {
    DFLASH_HIP_OK(hipFuncSetAttribute(k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, k.lds));
    done = true;
  }
  void* args[] = {&p};
  DFLASH_HIP_OK(hipLaunchKernel(k.fn, dim3((unsigned)(p.slices * p.lanes)), dim3(64 * kWaves), args, k.lds, stream));
  return DFLASH_OK;
}
}  // namespace dflash
