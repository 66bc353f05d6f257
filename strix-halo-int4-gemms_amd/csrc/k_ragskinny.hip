// Ragged forward with few rows a group: the skinny tiles of shk_skinny.h on
// the packed operands, one launch, no conversion (launch_f6_ragged_fwd picks
// it through ragged_skinny_rows).
//
// With a handful of tokens an expert the call is bound by reading the
// experts' weights once; the fp6 path reads them, writes them 1.5 times as
// large and reads those (64 experts of 1024 x 2048, 64 rows: 49.0 us a call,
// 16.3 here).  Here a workgroup streams one column tile of its
// group's packed B for 16, 32 or 64 rows of A.  It finds its rows itself, by
// a wave's scan of the group sizes, so no task list stands before it; one
// more workgroup builds the list that the call leaves to its caller.
#include <algorithm>
#include <cmath>

#include "shk_skinny.h"
#include "shk_table.h"

namespace shk {
namespace {

template <int LAYOUT, int R, bool SUBCH, int NW = SK_NW>
using C = SkCfg<4, LAYOUT, R, false, SUBCH, SUBCH ? 16 : 0, NW>;

// Group sizes as the kernel reads them: any int32 is taken as rows of
// [0, M], so that any sizes are safe (their check may still be running).
__device__ __forceinline__ int group_rows(const RaggedFwdArgs& p, int g) {
  return g < p.groups ? max(0, min(p.job.sizes[g], p.M)) : 0;
}
// Inclusive sum over the wave.
__device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(v, off, 64);
    if (lane >= off) v += y;
  }
  return v;
}

// Row task `task` of the groups' R-row blocks: its group, first row and the
// group's end.  False past the last task, or if it holds no row of A.
template <int R>
__device__ __forceinline__ bool find_rows(const RaggedFwdArgs& p, int task, int lane, int& group, int& row, int& end) {
  int first_row = 0, first_task = 0;
  for (int g0 = 0; g0 < p.groups; g0 += 64) {
    const int size = group_rows(p, g0 + lane);
    const int rows = wave_scan(size, lane), tasks = wave_scan((size + R - 1) / R, lane);
    const int total_tasks = __builtin_amdgcn_readlane(tasks, 63);
    if (task < first_task + total_tasks) {
      // the lane whose tasks hold it: the first with an inclusive sum past it
      const int l = __ffsll(__ballot(first_task + tasks > task)) - 1;
      const int lrows = __builtin_amdgcn_readlane(rows, l), lsize = __builtin_amdgcn_readlane(size, l);
      const int ltasks = __builtin_amdgcn_readlane(tasks, l);
      const int start = first_row + lrows - lsize, t0 = first_task + ltasks - (lsize + R - 1) / R;
      group = g0 + l;
      row = start + (task - t0) * R;
      end = min(start + lsize, p.M);
      return row < end;
    }
    first_task += total_tasks;
    // (saturates at M, past which no task holds a row)
    first_row = min(first_row + __builtin_amdgcn_readlane(rows, 63), p.M);
  }
  return false;
}

// The tasks of all groups.
template <int R>
__device__ __forceinline__ int count_tasks(const RaggedFwdArgs& p, int lane) {
  int n = 0;
  for (int g0 = 0; g0 < p.groups; g0 += 64) n += (group_rows(p, g0 + lane) + R - 1) / R;
  n = wave_scan(n, lane);
  return __builtin_amdgcn_readlane(n, 63);
}

template <class T>
__global__ __launch_bounds__(T::NT) void ragged_skinny_kernel(const RaggedFwdArgs p) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[T::LDS_BYTES];
  __shared__ int last_flag;
  if (blockIdx.x == gridDim.x - 1) {
    int* const scratch = reinterpret_cast<int*>(smem);
    static_assert(T::LDS_BYTES >= (int)sizeof(int) * (2 * (kFusedTaskGroups + 1) + T::NW), "task arrays fit");
    build_task_list<T::NT>(p.job, scratch, scratch + kFusedTaskGroups + 1, scratch + 2 * (kFusedTaskGroups + 1));
    return;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles_n = (p.N + T::BN - 1) / T::BN;
  const int units = min(count_tasks<T::R>(p, lane), ((int)gridDim.x - 1) / tiles_n) * tiles_n;
  if ((int)blockIdx.x >= units) return;
  // each XCD takes consecutive tasks with all their column tiles
  const int u = sk_xcd_remap(blockIdx.x, units);
  const int task = u / tiles_n, tn = u - task * tiles_n;
  int g, row, end;
  if (!find_rows<T::R>(p, task, lane, g, row, end)) return;
  DenseArgs q{};
  q.a = p.lhs;
  q.b = p.rhs + (long)g * (p.K / 2) * p.N;
  q.a_scale = p.a_scale;
  q.b_scale = p.b_scale + (long)g * (T::SUBCH ? p.scale_cols : 1) * p.N;
  q.out = p.out;
  q.M = end;
  q.N = q.b_cols = p.N;
  q.K = p.K;
  q.lda = p.lda;
  q.ldb = p.ldb;
  q.subchannel = p.subchannel;
  q.scale_cols = p.scale_cols;
  q.epilogue = EPI_NONE;
  q.out_mode = p.out_mode;
  if constexpr (T::SUBCH)
    sk_unit_sc<T, true>(q, smem, lane, wave, row, tn * T::BN);
  else
    sk_unit_pc<T, true, true>(q, smem, &last_flag, lane, wave, row, tn * T::BN, 0, 1, 0);
}

// Workgroups of a launch of tiles of `rows` rows and `bn` columns: every
// group's last block may be partial; one more builds the task list.
long workgroups(const RaggedFwdArgs& a, int rows, int bn) {
  return ((long)a.groups + a.M / rows) * ((a.N + bn - 1) / bn) + 1;
}
template <class T>
hipError_t launch(const RaggedFwdArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(ragged_skinny_kernel<T>, dim3((unsigned)workgroups(a, T::R, T::BN)), dim3(T::NT), 0, s, a);
  return hipGetLastError();
}

template <int LAYOUT>
hipError_t launch_rows(const RaggedFwdArgs& a, int rows, hipStream_t s) {
  if (a.subchannel > 0) {
    if (rows == 16 && a.subchannel >= 128) return launch<C<LAYOUT, 16, true, 8>>(a, s);
    return rows == 16 ? launch<C<LAYOUT, 16, true>>(a, s) : launch<C<LAYOUT, 32, true>>(a, s);
  }
  if (rows == 16) return launch<C<LAYOUT, 16, false>>(a, s);
  return rows == 32 ? launch<C<LAYOUT, 32, false>>(a, s) : launch<C<LAYOUT, 64, false>>(a, s);
}

// What the host knows is the rows of all groups, so the rule goes by their
// average r = M / groups, and by R-row tasks of groups * (r / R + 1/2).  Calls
// on the two paths, tasks and conversion included, rows drawn unevenly (us,
// skinny and fp6):
//  * per-channel, groups x N x K: r = 1: 64 x 1024 x 2048 16.3 (16 rows) and
//    49.0; r = 8: 8 x 1408 x 2048 7.7 and 25.9; r = 16: 16 x 4096^2 42.3 (32)
//    and 102.7; r = 64: 59.1 (64) and 110.4; r = 256: 136 and 152, 32 x
//    2048 x 1024 61 and 44, 64 x 1024 x 2048 82 and 80; r = 1024: 8 x 1408 x
//    2048 54.0 and 34.8.  Up to 24 rows every shape gains; above, the 64-row
//    tiles' time (7 ns + 4.6 ns per 1024 K a tile, and 6 us) stands against
//    the conversion's (5 TB/s) and the fp6 tiles' rounds.  Tiles of 16 rows
//    up to 12 (r = 16, 64 x 1024 x 2048: 21.7, 20.6 and 21.9 with 16, 32 and
//    64 rows; r = 32: 31.1, 25.6 and 22.5).
//  * groups of 128 along K: r = 8: 8 x 1408 x 2048 13.2 and 33.0; r = 32: 23.5
//    and 33.4; r = 64: 30.4 and 33.8; r = 1: 64 x 1024 x 2048 42.7 and 58.6;
//    r = 16: 61.6 and 62.7; r = 32: 85.6 and 63.9.  Groups of 32: r = 4: 64 x
//    1024 x 2048 89.8 and 104.6; r = 16: 131 and 105.
// The figures are fits to ragged calls, whose tiles find their rows and leave a
// list (the dense tiles' stand at sk_plan).  The path is taken where its
// prediction is 1.15 (subchannel 1.1) times shorter, since uneven groups make
// more tasks than the average does.
int predicted_rows(const RaggedFwdArgs& a) {
  const bool nt = a.layout == SHK_LAYOUT_NT;
  if (a.job.sizes == nullptr || a.groups > kFusedTaskGroups || (a.layout != SHK_LAYOUT_NN && !nt)) return 0;
  // 16-byte pieces of both operands, 32-bit offsets
  auto aligned16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (!aligned16(a.lhs) || !aligned16(a.rhs) || a.K < 32 || a.K % 32 || a.N % 16) return 0;
  if (a.M > 65536 || a.K > 65536 || (long)a.N * a.K > (1L << 32)) return 0;
  const double g = a.groups, n = a.N, k = a.K, r = a.M / g;
  const double convert = 6.0 + 2.5e-7 * (a.M + g * n) * k;
  auto tasks = [&](int rows) { return std::max(std::min(g, (double)a.M), g * (r / rows + 0.5)); };
  if (a.subchannel == 0) {
    if (r <= 24) return r <= 12 ? 16 : 32;
    const double rounds = std::ceil(g * (r / 128 + 0.5) * std::ceil(n / 128) / 256);
    const double fp6 = convert + 4.0 + 4.0e-3 * k + (2.6 + 2.0e-3 * k) * (rounds - 1);
    const double skinny = 6.0 + tasks(64) * std::ceil(n / 64) * (0.007 + 4.5e-6 * k);
    return 1.15 * skinny < fp6 ? 64 : 0;
  }
  const int i = a.subchannel == 32 ? 0 : (a.subchannel == 64 ? 1 : (a.subchannel == 128 ? 2 : 3));
  if (a.subchannel != (32 << i) || a.K % a.subchannel || r > 64) return 0;
  static constexpr double product[4] = {2.9e-8, 1.5e-8, 1.07e-8, 0.85e-8};
  static constexpr double fixed[4] = {5.0, 5.0, 5.0, 3.5}, per_k[4] = {0.0215, 0.0125, 0.0061, 0.0038};
  const double tiles = g * (std::floor(r / 128) + 1) * std::ceil(n / 128);
  const double fp6 = convert + (fixed[i] + per_k[i] * k) * (tiles <= 256 ? 1.0 : 1.3 * std::ceil(tiles / 512));
  const double low = 6.0 + 1.35 * product[i] * 16 * tasks(16) * n * k;
  const double high = 6.0 + product[i] * 32 * tasks(32) * n * k;
  return 1.1 * std::min(low, high) < fp6 ? (low <= high ? 16 : 32) : 0;
}

}  // namespace

// The predicted choice, unless its grid is more than a launch can hold: below
// 2^32 work-items, of at most 512 a workgroup (many experts with a very wide
// N; the fp6 tiles are 128 columns wide).
int ragged_skinny_rows(const RaggedFwdArgs& a) {
  const int rows = predicted_rows(a);
  const int bn = a.subchannel > 0 ? 16 : SK_BN, threads = rows == 16 && a.subchannel >= 128 ? 512 : 64 * SK_NW;
  return rows && workgroups(a, rows, bn) * threads < (1L << 32) ? rows : 0;
}

hipError_t launch_ragged_skinny(const RaggedFwdArgs& a, int rows, hipStream_t s) {
  return a.layout == SHK_LAYOUT_NT ? launch_rows<SHK_LAYOUT_NT>(a, rows, s) : launch_rows<SHK_LAYOUT_NN>(a, rows, s);
}

}  // namespace shk
