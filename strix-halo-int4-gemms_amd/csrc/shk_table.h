// Internal kernel-table plumbing shared by the kernel translation units and
// the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "../../include/strix_halo_gfx950.h"
#include "shk_i8.h"

namespace shk {

using DenseLaunchFn = hipError_t (*)(const DenseArgs&, dim3, hipStream_t);
using RaggedFwdLaunchFn = hipError_t (*)(const RaggedFwdArgs&, dim3, hipStream_t);
using RaggedBwdLaunchFn = hipError_t (*)(const RaggedBwdArgs&, dim3, hipStream_t);

struct Entry {
  shk_kernel_desc d;
  DenseLaunchFn dense;
  RaggedFwdLaunchFn fwd;
  RaggedBwdLaunchFn bwd;
  DenseLaunchFn converted;  // fp6 entries: the GEMM alone, on converted operands
};

template <class C>
hipError_t launch_dense_t(const DenseArgs& a, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL(dense_gemm_kernel<C>, grid, dim3(C::NT), 0, s, a);
  return hipGetLastError();
}
// fp6 path.  f6_convert_operand converts A (operand 0) or B (operand 1) of
// a dense call into its part of the workspace (A first, then B); the GEMM
// then reads both parts.
// (The FP6 entries' M, b_cols and K are tile multiples, which the padding
// leaves as they are; the FP6_EDGE entries' are not.)
inline uint8_t* f6_work_b(const DenseArgs& a) {
  return a.work + f6_operand_bytes(f6_pad_rows(a.M), f6_pad_k(a.K));
}
inline F6PackArgs f6_pack_args(const DenseArgs& a, int operand, bool swiglu) {
  const int kb = (int)(f6_pad_k(a.K) / 64);
  // dense operands are validated 16-byte aligned
  if (operand == 0) return F6PackArgs{a.a, a.work, a.lda, a.M, kb, 0, 1, 0, 0, nullptr, a.K, 16};
  return F6PackArgs{a.b, f6_work_b(a), a.ldb, a.b_cols, kb, swiglu ? a.N : 0, 1, 0, 0, nullptr, a.K, 16};
}
inline bool f6_mn_major(const DenseArgs& a, int operand) {
  return operand == 0 ? a.layout == SHK_LAYOUT_TN : a.layout != SHK_LAYOUT_NT;
}
inline hipError_t f6_convert_operand(const DenseArgs& a, int operand, bool swiglu, hipStream_t s) {
  return launch_f6_pack(f6_pack_args(a, operand, swiglu), f6_mn_major(a, operand), s);
}
// How an FP6_EDGE per-channel call runs: 128 x 128 tiles in rings of `slots`
// (plain epilogues), or, with slots 0, 256-row tiles of which the last
// `half_columns` column tiles run as 128-row tiles; `tiles` workgroups.
//
// The 256-row tile reads half the bytes per product, one workgroup a CU; the
// small one fills the chip on small grids and has a short epilogue.  Both
// costs are fits to a sweep of M 192..8176 over N x K of 1024 x 4096, 4096 x
// 1024, 4096^2, 11008 x 4096, 16384 x 4096 and 8192^2 (us): a round of 256
// large tiles 14 + 4.9 K/1024, 256 small tiles 2.6 + 2.05 K/1024.  Measured
// on both sides of the line, call with conversion, small and large tiles:
// 1008 x 4096^2 26.1 and 31.6 us, 4160 x 4096 x 1024 30.6 and 37.7, 1008 x
// 11008 x 4096 46.9 and 47.0, 1008 x 16384 x 4096 64.0 and 58.7, 8176 x
// 8192^2 369 and 295.
//
// Half-height tiles run a partial last round in about 0.6 of its time where
// all of them fit one round of the chip: 1008 x 11008 x 4096 SwiGLU, 344
// tiles, 85.3 -> 80.2 us; 512 x 4096^2 SwiGLU, 64 tiles, 39.7 -> 31.8.
struct F6EdgePlan {
  int slots;
  int half_columns;
  long tiles;
  double us;  // the GEMM's predicted time
};
constexpr long kF6EdgeCus = 256;
inline F6EdgePlan f6_edge_plan(long m, long n, long k, bool swiglu) {
  const double k1 = (double)k / 1024.0;
  const long bn = swiglu ? 128 : 256;
  const long tm = (m + 255) / 256, tn = (n + bn - 1) / bn, tm2 = (m + 127) / 128;
  const long tiles = tm * tn, rounds = tiles / kF6EdgeCus, rest = tiles % kF6EdgeCus;
  const double round_us = 14.0 + 4.9 * k1;
  F6EdgePlan p{0, 0, tiles, round_us * (double)(rounds + (rest > 0 ? 1 : 0))};
  if (rest > 0) {
    const long c = rounds == 0 ? tn : (rest + tm - 1) / tm;
    if (tm2 * c <= kF6EdgeCus) {
      p.half_columns = (int)c;
      p.tiles = tm * (tn - c) + tm2 * c;
      p.us = round_us * ((double)rounds + 0.6);
    }
  }
  if (!swiglu) {
    const long small = tm2 * ((n + 127) / 128);
    const double us = (2.6 + 2.05 * k1) * (double)((small + kF6EdgeCus - 1) / kF6EdgeCus);
    if (us <= p.us) p = F6EdgePlan{small <= 2 * kF6EdgeCus ? 3 : 2, 0, small, us};
  }
  return p;
}

// Large-K per-channel fp6 calls (K > F6_MAX_K): the int32 sums of the K
// slices go to the workspace past both converted operands, [M, b_cols]
// int32, which f6_large_k_begin clears and f6_large_k_end turns into the
// output (scales and epilogue, or the raw sums) (k_f6.hip).
inline int32_t* f6_large_k_acc(const DenseArgs& a) {
  return reinterpret_cast<int32_t*>(a.work + f6_operand_bytes(a.M, a.K) + f6_operand_bytes(a.b_cols, a.K));
}
hipError_t f6_large_k_begin(const DenseArgs& a, hipStream_t s);
hipError_t f6_large_k_end(const DenseArgs& a, bool swiglu, hipStream_t s);

template <class C>
hipError_t launch_f6_gemm_t(const DenseArgs& a, dim3 grid, hipStream_t s) {
  DenseArgs g = a;
  g.a = a.work;
  g.b = a.work + f6_operand_bytes(a.M, a.K);
  if (a.K > F6_MAX_K) {
    hipError_t err = f6_large_k_begin(a, s);
    if (err != hipSuccess) return err;
    g.out = f6_large_k_acc(a);
    const unsigned slices = (unsigned)((a.K + F6_MAX_K - 1) / F6_MAX_K);
    hipLaunchKernelGGL((f6_gemm_kernel<C, OUT_I32_ADD, EPI_NONE>), dim3(grid.x, slices), dim3(256), 0, s, g);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    return f6_large_k_end(a, C::SWIGLU, s);
  }
  if (a.out_mode == OUT_I32) {
    hipLaunchKernelGGL((f6_gemm_kernel<C, OUT_I32, EPI_NONE>), grid, dim3(256), 0, s, g);
  } else if (a.out_mode == OUT_F32) {
    if (!C::SWIGLU && a.epilogue == EPI_RELU2)
      hipLaunchKernelGGL((f6_gemm_kernel<C, OUT_F32, EPI_RELU2>), grid, dim3(256), 0, s, g);
    else
      hipLaunchKernelGGL((f6_gemm_kernel<C, OUT_F32, EPI_NONE>), grid, dim3(256), 0, s, g);
  } else if (!C::SWIGLU && a.epilogue == EPI_RELU2) {
    hipLaunchKernelGGL((f6_gemm_kernel<C, OUT_BF16, EPI_RELU2>), grid, dim3(256), 0, s, g);
  } else {
    hipLaunchKernelGGL((f6_gemm_kernel<C, OUT_BF16, EPI_NONE>), grid, dim3(256), 0, s, g);
  }
  return hipGetLastError();
}
template <class C>
hipError_t launch_f6_t(const DenseArgs& a, dim3 grid, hipStream_t s) {
  hipError_t err = launch_f6_pack2(f6_pack_args(a, 0, C::SWIGLU), f6_mn_major(a, 0), f6_pack_args(a, 1, C::SWIGLU),
                                   f6_mn_major(a, 1), s, nullptr, true);
  if (err == hipSuccess) err = launch_f6_gemm_t<C>(a, grid, s);
  return err;
}
// Workgroups of a persistent launch of `kernel` with `block` threads: its
// resident slots on the current device (occupancy x CUs), rounded down to a
// multiple of 8 so that a workgroup keeps its XCD, and at most `tiles`
// (capi.hip).
hipError_t persistent_grid(const void* kernel, int block, unsigned tiles, unsigned* grid);
template <auto K>
hipError_t launch_persistent(const DenseArgs& g, unsigned tiles, int block, hipStream_t s) {
  unsigned n = 0;
  const hipError_t err = persistent_grid(reinterpret_cast<const void*>(K), block, tiles, &n);
  if (err != hipSuccess) return err;
  void* args[] = {const_cast<DenseArgs*>(&g)};
  return hipLaunchKernel(reinterpret_cast<const void*>(K), dim3(n), dim3(block), args, 0, s);
}
// fp6 GEMM on converted operands, persistent schedule (plain epilogues).
template <class C>
hipError_t launch_f6_gemm_persistent_t(const DenseArgs& a, dim3 grid, hipStream_t s) {
  static_assert(!C::SWIGLU, "persistent entries are plain");
  DenseArgs g = a;
  g.a = a.work;
  g.b = a.work + f6_operand_bytes(a.M, a.K);
  const bool relu2 = a.epilogue == EPI_RELU2;
  if (a.out_mode == OUT_I32) return launch_persistent<&f6_gemm_persistent<C, OUT_I32, EPI_NONE>>(g, grid.x, 256, s);
  if (a.out_mode == OUT_F32)
    return relu2 ? launch_persistent<&f6_gemm_persistent<C, OUT_F32, EPI_RELU2>>(g, grid.x, 256, s)
                 : launch_persistent<&f6_gemm_persistent<C, OUT_F32, EPI_NONE>>(g, grid.x, 256, s);
  return relu2 ? launch_persistent<&f6_gemm_persistent<C, OUT_BF16, EPI_RELU2>>(g, grid.x, 256, s)
               : launch_persistent<&f6_gemm_persistent<C, OUT_BF16, EPI_NONE>>(g, grid.x, 256, s);
}
template <class C>
hipError_t launch_f6_persistent_t(const DenseArgs& a, dim3 grid, hipStream_t s) {
  hipError_t err = launch_f6_pack2(f6_pack_args(a, 0, false), f6_mn_major(a, 0), f6_pack_args(a, 1, false),
                                   f6_mn_major(a, 1), s, nullptr, true);
  if (err == hipSuccess) err = launch_f6_gemm_persistent_t<C>(a, grid, s);
  return err;
}
template <class C>
hipError_t launch_dense_persistent_t(const DenseArgs& a, dim3 grid, hipStream_t s) {
  return launch_persistent<&dense_gemm_persistent<C>>(a, grid.x, C::NT, s);
}
// int8 32x32 engine: one kernel per output mode and epilogue.  A grid of
// 256-row tiles (K-major A) whose last round of workgroups would be partial
// runs the column tiles of that round as 128-row tiles, twice as many and
// half as long, when they fit one round (i8_gemm_kernel).
template <class C, int MODE, int EPI>
hipError_t launch_i8_k(const DenseArgs& a, dim3 grid, hipStream_t s) {
  auto* k = &i8_gemm_kernel<C, MODE, EPI>;
  DenseArgs g = a;
  g.split_tn = 0;
  if constexpr (C::BM == 256 && C::A_KMAJOR) {
    const long tiles_m = a.M / C::BM, tiles_n = a.N / C::BN;
    unsigned slots = 0;
    const hipError_t err = persistent_grid(reinterpret_cast<const void*>(k), 256, 0xFFFFFFFFu, &slots);
    if (err != hipSuccess) return err;
    const long tiles = tiles_m * tiles_n;
    const long rest = slots > 0 ? tiles % slots : 0;
    if (tiles > (long)slots && rest > 0) {
      const long c = (rest + tiles_m - 1) / tiles_m;  // trailing column tiles holding the partial round
      if (2 * tiles_m * c <= (long)slots && c < tiles_n) {
        g.split_tn = (int)(tiles_n - c);
        grid = dim3((unsigned)(tiles_m * (tiles_n - c) + 2 * tiles_m * c));
      }
    }
  }
  hipLaunchKernelGGL(k, grid, dim3(256), 0, s, g);
  return hipGetLastError();
}
template <class C>
hipError_t launch_i8_t(const DenseArgs& a, dim3 grid, hipStream_t s) {
  if (a.out_mode == OUT_I32) return launch_i8_k<C, OUT_I32, EPI_NONE>(a, grid, s);
  if (a.out_mode == OUT_F32) {
    if (!C::SWIGLU && a.epilogue == EPI_RELU2) return launch_i8_k<C, OUT_F32, EPI_RELU2>(a, grid, s);
    return launch_i8_k<C, OUT_F32, EPI_NONE>(a, grid, s);
  }
  if (!C::SWIGLU && a.epilogue == EPI_RELU2) return launch_i8_k<C, OUT_BF16, EPI_RELU2>(a, grid, s);
  return launch_i8_k<C, OUT_BF16, EPI_NONE>(a, grid, s);
}
template <class C>
hipError_t launch_fwd_t(const RaggedFwdArgs& a, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL(ragged_fwd_kernel<C>, grid, dim3(C::NT), 0, s, a);
  return hipGetLastError();
}
template <class C>
hipError_t launch_bwd_t(const RaggedBwdArgs& a, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL(ragged_bwd_kernel<C>, grid, dim3(C::NT), 0, s, a);
  return hipGetLastError();
}

template <class C>
constexpr shk_kernel_desc desc_of(int family, int layout, int group_m) {
  return shk_kernel_desc{
      -1,
      family,
      C::BITS,
      layout,
      C::SUBCH ? SHK_SCALE_SUBCHANNEL : SHK_SCALE_PER_CHANNEL,
      C::SUBCH ? (C::MK == 32 ? 32 : 64) : 0,
      C::SUBCH ? (C::MK == 32 ? 32 : 256) : 0,
      C::SWIGLU ? SHK_EPI_KIND_SWIGLU : SHK_EPI_KIND_PLAIN,
      C::BM,
      C::BN,
      C::BK,
      C::NT / 64,
      C::NUM_STAGES,
      C::LDS_BYTES,
      group_m,
      SHK_OPERANDS_PACKED,
      SHK_SCHEDULE_STANDARD,
      1,
  };
}

template <class C>
Entry dense_entry(int layout, int group_m) {
  return Entry{desc_of<C>(SHK_FAMILY_DENSE, layout, group_m), &launch_dense_t<C>, nullptr, nullptr, nullptr};
}
template <class C>
Entry i8_entry(int layout, int group_m) {
  static_assert(C::LDS_BYTES == I8Engine<C>::LDS_BYTES && C::NUM_STAGES == I8Engine<C>::P, "table geometry");
  shk_kernel_desc d = desc_of<C>(SHK_FAMILY_DENSE, layout, group_m);
  d.lds_bytes += MFMA32_SCALE_BYTES;
  return Entry{d, &launch_i8_t<C>, nullptr, nullptr, nullptr};
}
template <class C>
Entry f6_entry(int layout) {
  shk_kernel_desc d = desc_of<C>(SHK_FAMILY_DENSE, layout, 8);
  d.num_stages = F6Engine<C>::P;
  d.lds_bytes = F6Engine<C>::LDS_BYTES + MFMA32_SCALE_BYTES;
  d.operand_format = SHK_OPERANDS_FP6;
  return Entry{d, &launch_f6_t<C>, nullptr, nullptr, &launch_f6_gemm_t<C>};
}
// Persistent-schedule entries of the same kernels.
template <class C>
Entry f6_persistent_entry(int layout) {
  Entry e = f6_entry<C>(layout);
  e.d.schedule = SHK_SCHEDULE_PERSISTENT;
  e.dense = &launch_f6_persistent_t<C>;
  e.converted = &launch_f6_gemm_persistent_t<C>;
  return e;
}
template <class C>
Entry dense_persistent_entry(int layout, int group_m) {
  Entry e = dense_entry<C>(layout, group_m);
  e.d.schedule = SHK_SCHEDULE_PERSISTENT;
  e.dense = &launch_dense_persistent_t<C>;
  return e;
}
// Split-K entries of a dense tile: grid.y = split, each workgroup sums one
// K slice and adds its scaled fp32 partial into the zeroed output.
template <class C>
Entry split_entry(int layout, int group_m, int split) {
  Entry e = dense_entry<C>(layout, group_m);
  e.d.split_k = split;
  return e;
}
template <class C>
Entry fwd_entry(int layout) {
  return Entry{desc_of<C>(SHK_FAMILY_RAGGED_FWD, layout, 1), nullptr, &launch_fwd_t<C>, nullptr, nullptr};
}
template <class C>
Entry bwd_entry(int layout) {
  return Entry{desc_of<C>(SHK_FAMILY_RAGGED_BWD, layout, 1), nullptr, nullptr, &launch_bwd_t<C>, nullptr};
}

// Skinny entries (SHK_OPERANDS_STREAM, shk_skinny.h).  Workgroups that share
// a per-channel tile's K: enough to give about kSkTargetUnits workgroups (one
// per CU of an MI355X; at M = 16, N = K = 8192 two workgroups per tile run
// 8.8 us against 9.9 us for four, each K split adding a tail of device-scope
// round trips) while every wave keeps at least two stages, at most 16;
// and for int4 at least as many as keep each wave's x256 int32 sum within
// 1023 stages of 128 K (up to 64 at K = 2^24).  Subchannel tiles always use
// one.
constexpr int kSkTargetUnits = 256;
inline int sk_needed_splits(int bits, long k) {
  long need = 1;
  if (bits == 4)
    while (need * 4L * 1023L < (k + 127) / 128) need *= 2;
  return (int)need;
}
inline int sk_splits(int bits, long tiles, long k) {
  const long nst = bits == 4 ? (k + 127) / 128 : (k + 63) / 64;
  long s = 1;
  while (s * 2 <= 16 && tiles * s * 2 <= kSkTargetUnits && nst >= 16L * s) s *= 2;
  const long need = sk_needed_splits(bits, k);
  return (int)(s > need ? s : need);
}

// Whether a skinny entry plans its tiles' rows for each call (k_skinny.hip
// sk_rows_entry); the other entries' tiles are block_m rows.
inline bool sk_plans_rows(const shk_kernel_desc& d) {
  return d.operand_format == SHK_OPERANDS_STREAM && d.group_size_m > 1;
}
// The tile rows such an entry takes for a call of M rows: 16, 32 or 64,
// masked to M (subchannel 16 or 32).  A taller tile reads B fewer times and
// keeps the matrix cores busier per byte; a lower one gives a small N more
// workgroups and computes fewer rows that are not there.
//
// The height of the smallest predicted time, but the tallest that divides M
// where that is within 5%, the fits' own error: whole tiles need no mask and
// a height that changes little is not worth a wrong guess.  The time (us) is
// linear in what a launch of u workgroups, each with w = K / 4096 of its part
// of K and g = K / 32 groups, takes on 256 CUs: one round, whether there is a
// second, how many whole rounds of 256 and of 512 (two a CU), the workgroups
// past the first 256, MN-major A and B (16-byte pieces of a row an
// instruction), and the doublings of K's split.  Fitted to 4500 calls drawn
// over M 16..8192, N 512..16384, K 512..14336 in all layouts and widths,
// every height measured: median error 4%, a tenth above 11%.  Measured, 16,
// 32 and 64 rows: int8 SwiGLU 48 x 11008 x 4096 NT 29.9, 32.5, 25.7 us; 288 x
// 1088 x 4480 with A MN-major 28.8, 20.0 and 24.5; int4 SwiGLU 64 x 12224 x
// 6208 31.6, 32.0, 25.4; int4 plain 112 x 8192^2 27.7, 21.9, 17.7; 32 x 10688
// x 12224 22.7, 17.0.  16 and 32 rows, groups of 128: 400 x 4096^2 110 and 80
// us, 48 x 16064 x 5120 NT 46.5 and 53.0.
struct SkPlan {
  int rows;
  double us;
};
constexpr int kSkTerms = 9;      // constant, w, w rounds, w double rounds, w second, past, rounds, A MN, log2 splits
constexpr int kSkSubTerms = 10;  // constant, w, g, w and g double rounds, w and g second, past, A MN, B MN
// [8-bit][SwiGLU][16, 32, 64 rows]
constexpr double kSkFit[2][2][3][kSkTerms] = {
    {{{3.76, 2.96, 0.96, 3.11, 0.2, 0.77, 0.1, 1.39, 0.88},
       {3.91, 4.12, 1.8, 2.72, 0.16, 0.54, 0.65, 1.07, 1.19},
       {4.89, 5.84, 2.69, 3.29, 0.33, 1.19, 0.64, 0.1, 1.64}},
      {{3.91, 5.25, 4.09, 1.05, 0.67, 0.92, 0.07, 1.09, 1.19},
       {4.97, 6.96, 6.16, 0.83, 1.12, 0.51, 3.21, 0.32, 1.55},
       {6.94, 9.81, 8.75, 0.0, 0.81, 0.14, 5.91, 1.36, 2.78}}},
     {{{3.71, 3.68, 4.83, 0.45, 0.0, 0.41, 0.0, 3.55, 1.02},
       {3.64, 5.78, 5.15, 2.5, 0.0, 0.55, 0.0, 3.24, 1.09},
       {4.16, 8.21, 7.34, 4.93, 0.0, 0.77, 0.0, 2.21, 1.59}},
      {{2.87, 10.23, 6.51, 4.32, 1.34, 0.51, 0.0, 3.5, 1.14},
       {3.74, 11.02, 7.83, 4.71, 2.69, 0.0, 2.68, 3.73, 1.71},
       {5.52, 14.08, 12.06, 1.6, 1.05, 0.14, 4.59, 2.99, 2.72}}}};
// [8-bit][SwiGLU][groups of a stage or more][16, 32 rows]
constexpr double kSkSubFit[2][2][2][2][kSkSubTerms] = {
    {{{{3.5, 2.26, 3.42, 2.89, 3.49, 1.45, 0.15, 0.89, 0.44, 0.13},
       {3.48, 0.06, 6.6, 0.44, 6.75, 1.04, 0.47, 0.98, 0.0, 0.05}},
      {{3.63, 1.63, 1.64, 2.68, 1.95, 0.89, 0.77, 0.72, 1.53, 0.6},
       {3.84, 4.06, 3.62, 4.79, 3.72, 1.07, 0.55, 1.02, 0.79, 0.37}}},
     {{{3.84, 0.47, 6.04, 0.29, 6.52, 0.39, 0.71, 1.01, 0.96, 0.62},
       {3.78, 0.14, 10.11, 0.68, 10.49, 0.0, 1.15, 1.06, 0.74, 0.64}},
      {{4.0, 3.09, 4.1, 5.12, 3.22, 1.21, 0.64, 0.97, 2.21, 1.16},
       {3.86, 4.44, 6.46, 6.36, 5.75, 2.24, 0.0, 1.03, 1.13, 0.8}}}},
    {{{{3.59, 0.0, 3.86, 0.0, 4.24, 0.0, 0.56, 0.91, 1.52, 0.59},
       {3.41, 0.0, 5.68, 0.0, 6.02, 0.0, 0.84, 0.94, 1.15, 0.48}},
      {{3.42, 2.59, 1.44, 4.91, 1.73, 1.86, 0.55, 0.57, 4.23, 1.94},
       {3.84, 5.39, 3.26, 9.06, 2.89, 2.21, 0.0, 0.84, 2.47, 1.64}}},
     {{{3.86, 0.0, 5.44, 0.0, 5.84, 0.0, 0.82, 1.02, 2.57, 0.75},
       {3.38, 0.0, 9.69, 0.0, 10.3, 0.0, 1.15, 0.91, 3.97, 1.54}},
      {{3.9, 4.15, 2.68, 9.52, 1.89, 2.21, 1.68, 0.63, 6.05, 4.11},
       {3.31, 6.32, 6.61, 11.59, 3.82, 2.14, 0.0, 0.74, 5.02, 3.92}}}}};
// `sub`: the group size, or 0 for per-channel scales.
inline SkPlan sk_plan(int bits, int sub, bool swiglu, int layout, long m, long n, long k) {
  const double a_mn = layout == SHK_LAYOUT_TN ? 1.0 : 0.0, b_mn = layout == SHK_LAYOUT_NN ? 1.0 : 0.0;
  SkPlan best{16, -1.0}, whole{16, -1.0};
  for (int i = 0; i < (sub > 0 ? 2 : 3); ++i) {
    const int rows = 16 << i;
    if (i > 0 && m <= rows / 2) break;
    // (where the K of one workgroup is bounded every tile keeps partials: no
    // more of them than M has rows, so that the workspace fits where it did)
    if (sub == 0 && m % rows != 0 && sk_needed_splits(bits, k) > 1) continue;
    const long tiles = (m + rows - 1) / rows * (sub > 0 ? n / 16 : n / 64);
    const int s = sub > 0 ? 1 : sk_splits(bits, tiles, k);
    const double u = (double)(tiles * s), w = (double)k / (double)s / 4096.0;
    const bool second = tiles * s > 256;
    const double past = second ? u / 256.0 - 1.0 : 0.0, wm = w * (1.0 + past), w2 = second ? w : 0.0;
    const double twice = (double)((tiles * s - 1) / 512);  // double rounds past the first
    double us = 0.0;
    if (sub > 0) {
      const double g = (double)k / (double)sub / 32.0;
      const double x[kSkSubTerms] = {1.0, w, g, w * twice, g * twice, w2, second ? g : 0.0, past, wm * a_mn, wm * b_mn};
      const double* f = kSkSubFit[bits == 8][swiglu][sub >= (bits == 4 ? 128 : 64)][i];
      for (int j = 0; j < kSkSubTerms; ++j) us += f[j] * x[j];
    } else {
      int halvings = 0;
      while ((1 << halvings) < s) ++halvings;
      const double rounds = (double)((tiles * s - 1) / 256);
      const double x[kSkTerms] = {1.0, w, w * rounds, w * twice, w2, past, rounds, wm * a_mn, (double)halvings};
      for (int j = 0; j < kSkTerms; ++j) us += kSkFit[bits == 8][swiglu][i][j] * x[j];
    }
    if (best.us < 0.0 || us < best.us) best = SkPlan{rows, us};
    if (m % rows == 0) whole = SkPlan{rows, us};
  }
  return whole.us <= 1.05 * best.us ? whole : best;
}
// Rows of a table entry's tiles.
inline int sk_tile_rows(const shk_kernel_desc& d, long m, long n, long k, int sub) {
  if (!sk_plans_rows(d)) return d.block_m;
  return sk_plan(d.dtype_bits, sub, d.epilogue_kind == SHK_EPI_KIND_SWIGLU, d.layout, m, n, k).rows;
}
// A skinny call: its tile rows, the workgroups sharing a tile's K (subchannel
// tiles always one), and with more than one split its workspace: the tiles' arrival counters, padded
// to 256 bytes, then an exact int32 partial of every (tile, split).  All of
// it is zero before the first launch and every launch leaves what it used
// zero, whatever the shapes of the launches that share it.
struct SkCall {
  int rows, splits;
  unsigned long long counter_bytes, workspace_bytes;  // 0 unsplit
};
// `sub`: the call's group size (0 per-channel; the workspace does not depend
// on it).
inline SkCall sk_call(const shk_kernel_desc& d, long m, long n, long k, int sub) {
  SkCall c{sk_tile_rows(d, m, n, k, sub), 1, 0, 0};
  if (d.scale_mode == SHK_SCALE_SUBCHANNEL) return c;
  const long tiles = ((m + c.rows - 1) / c.rows) * (n / d.block_n);
  c.splits = sk_splits(d.dtype_bits, tiles, k);
  if (c.splits > 1) {
    const long cf = d.epilogue_kind == SHK_EPI_KIND_SWIGLU ? 2 : 1;
    c.counter_bytes = (unsigned long long)((tiles * 4 + 255) & ~255L);
    // per (tile, split): (block_n / 16) output column tiles x (rows / 16) row
    // tiles x (up, gate) x 1 KiB
    c.workspace_bytes =
        c.counter_bytes + (unsigned long long)tiles * c.splits * (d.block_n / 16) * (c.rows / 16) * cf * 1024;
  }
  return c;
}

// Splits of the same call without a workspace: one, or 0 when K needs more.
inline int sk_direct_splits(const shk_kernel_desc& d, long k) {
  return d.scale_mode == SHK_SCALE_SUBCHANNEL || sk_needed_splits(d.dtype_bits, k) == 1 ? 1 : 0;
}

// Each kernel translation unit appends its entries in a fixed order
// (append_dense_f6(layout), append_dense_dma_<bits>_<layout>,
// append_dense_<bits>_<layout>, append_ragged_<layout>).
void append_dense_f6(std::vector<Entry>& t, int layout);
// fp6 entries for shapes that are no multiple of the fp6 tiles (k_f6edge.hip),
// after the skinny entries.
void append_edge_f6(std::vector<Entry>& t, int layout);
void append_dense_dma_4_0(std::vector<Entry>& t);
void append_dense_dma_4_1(std::vector<Entry>& t);
void append_dense_dma_4_2(std::vector<Entry>& t);
void append_dense_dma_8_0(std::vector<Entry>& t);
void append_dense_dma_8_1(std::vector<Entry>& t);
void append_dense_dma_8_2(std::vector<Entry>& t);
void append_dense_4_0(std::vector<Entry>& t);
void append_dense_4_1(std::vector<Entry>& t);
void append_dense_4_2(std::vector<Entry>& t);
void append_dense_8_0(std::vector<Entry>& t);
void append_dense_8_1(std::vector<Entry>& t);
void append_dense_8_2(std::vector<Entry>& t);
// Persistent-schedule int4 entries (plain epilogue kind), appended after
// the ragged families: the fp6 per-channel and subchannel tiles
// (append_persistent_f6(layout)) and the register-staged 64 x 64
// subchannel tiles for groups of 64 and 32 (append_persistent_4_<layout>).
void append_persistent_f6(std::vector<Entry>& t, int layout);
void append_persistent_4_0(std::vector<Entry>& t);
void append_persistent_4_1(std::vector<Entry>& t);
void append_persistent_4_2(std::vector<Entry>& t);
// Split-K 2/4/8 entries of the 128x128 per-channel tile (int4, int8) and of
// the 64x64 subchannel tiles (int4), per layout (append_split_<bits>_<layout>).
void append_split_4_0(std::vector<Entry>& t);
void append_split_4_1(std::vector<Entry>& t);
void append_split_4_2(std::vector<Entry>& t);
void append_split_8_0(std::vector<Entry>& t);
void append_split_8_1(std::vector<Entry>& t);
void append_split_8_2(std::vector<Entry>& t);
// Skinny entries per (bits, layout) (k_skinny.hip): for block_m 16, 32, 64
// the per-channel and subchannel tiles, plain and SwiGLU; for int4 the
// persistent plain tiles, split-K 1/2/4/8; then split-K 2/4/8 plain tiles.
void append_skinny_4_0(std::vector<Entry>& t);
void append_skinny_rows_4_0(std::vector<Entry>& t);
void append_skinny_4_1(std::vector<Entry>& t);
void append_skinny_rows_4_1(std::vector<Entry>& t);
void append_skinny_4_2(std::vector<Entry>& t);
void append_skinny_rows_4_2(std::vector<Entry>& t);
void append_skinny_8_0(std::vector<Entry>& t);
void append_skinny_rows_8_0(std::vector<Entry>& t);
void append_skinny_8_1(std::vector<Entry>& t);
void append_skinny_rows_8_1(std::vector<Entry>& t);
void append_skinny_8_2(std::vector<Entry>& t);
void append_skinny_rows_8_2(std::vector<Entry>& t);
void append_ragged_0(std::vector<Entry>& t);
void append_ragged_1(std::vector<Entry>& t);
void append_ragged_2(std::vector<Entry>& t);
void append_ragged_3(std::vector<Entry>& t);
int max_info_groups();
// fp6 ragged entries of one layout (k_f6ragged.hip): the forward (task
// tile 128) and the K-ragged backward, each per-channel and subchannel.
Entry f6_ragged_fwd_entry(int layout);
// Rows of the skinny tiles that a ragged forward runs in place of the fp6
// ones (k_ragskinny.hip), or 0.
int ragged_skinny_rows(const RaggedFwdArgs& a);
hipError_t launch_ragged_skinny(const RaggedFwdArgs& a, int rows, hipStream_t s);
Entry f6_ragged_sub_fwd_entry(int layout);
Entry f6_ragged_bwd_entry(int layout);
Entry f6_ragged_sub_bwd_entry(int layout);
// Workspace bytes of the fp6 ragged paths.
unsigned long long f6_ragged_fwd_workspace(int m, int n, int k, int groups, bool subchannel);
unsigned long long f6_ragged_bwd_workspace(int m, int n, int k_cap, int groups, bool subchannel);

// Non-table kernels (ragged.hip).
hipError_t launch_group_info(const int32_t* sizes, int groups, int tile, int align, int capacity,
                             int32_t* tasks, int32_t* num_tasks, int64_t* info, hipStream_t s);
hipError_t launch_bwd_finalize(float* out, const uint16_t* a_scale, const uint16_t* b_scale, int groups,
                               int m, int n, hipStream_t s);

}  // namespace shk
