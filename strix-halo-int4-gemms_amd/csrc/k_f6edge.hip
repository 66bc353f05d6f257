// FP6_EDGE entries (SHK_OPERANDS_FP6_EDGE): int4 shapes that are no multiple
// of the fp6 tiles.  M and N are multiples of 16 and 64, K of 32 (subchannel:
// of 64 and the group).  Same conversion and MFMA tiles as the FP6 entries;
// the converted operands are padded to whole 32-row panels and 128-K stages,
// and the stores stop at M and N.  Compiled like k_f6.hip.
#include "shk_f6small.h"
#include "shk_f6sub.h"
#include "shk_table.h"

namespace shk {
namespace {

template <int BN, bool SWIGLU>
using C = Cfg<4, true, true, 256, BN, 128, 2, 2, SWIGLU, false, 64, false, 0>;

// Per-channel 128 x 128 tile (shk_f6small.h): P ring slots, so three
// workgroups a CU with two slots and two with three.  One workgroup alone on
// a CU waits for its loads at every second stage with two slots: 256 tiles
// of K = 4096 (1008 x 4096) 31.3 us a call, with three slots 26.1; from 384
// tiles on two and three are within 2%.
using CSmall = Cfg<4, true, true, 128, 128, 128, 2, 2, false, false, 64, false, 0>;

template <int MODE, int EPI, int P>
__global__ __launch_bounds__(256, P == 2 ? 3 : 2) void f6_small_edge_kernel(const DenseArgs p) {
  using E = F6SmallEngine<CSmall, P>;
  __shared__ __attribute__((aligned(16))) uint8_t smem[E::LDS_BYTES + MFMA32_SCALE_BYTES];
  int tm, tn;
  dense_tile_coords(blockIdx.x, (p.M + 127) / 128, (p.N + 127) / 128, p.group_m, tm, tn);
  const int m0 = 128 * tm, n0 = 128 * tn;
  const int kpad = (int)f6_pad_k(p.K);
  E e;
  e.setup(smem, p.a, p.b, m0, n0, kpad / 64, f6_operand_bytes(f6_pad_rows(p.M), kpad),
          f6_operand_bytes(f6_pad_rows(p.N), kpad));
  float sa[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    sa[i] = MODE == OUT_I32 ? 0.0f : load_bf16(p.a_scale + min(m0 + e.out_row(i), p.M - 1));
  const OutView o{p.out, p.b_scale, p.N, p.M, p.N, 0, p.M, p.N};
  mfma32_prefetch_b_scales<CSmall, MODE, true>(e, o, n0, e.lds0 + E::LDS_BYTES + 256u * e.wave);
  e.run(kpad / 128);
  f6s_finish<MODE, true, EPI>(e, o, smem, m0, n0, sa);
}

template <bool SWIGLU, int MODE, int EPI>
void launch_edge(const DenseArgs& a, hipStream_t s) {
  constexpr int BN = SWIGLU ? 128 : 256;
  DenseArgs g = a;
  const int tiles_n = (g.N + BN - 1) / BN;
  const F6EdgePlan plan = f6_edge_plan(g.M, g.N, g.K, SWIGLU);
  if constexpr (!SWIGLU) {
    if (plan.slots) {
      const dim3 grid((unsigned)plan.tiles);
      if (plan.slots == 2) hipLaunchKernelGGL((f6_small_edge_kernel<MODE, EPI, 2>), grid, dim3(256), 0, s, g);
      else hipLaunchKernelGGL((f6_small_edge_kernel<MODE, EPI, 3>), grid, dim3(256), 0, s, g);
      return;
    }
  }
  g.split_tn = tiles_n - plan.half_columns;
  hipLaunchKernelGGL((f6_edge_gemm<C<BN, SWIGLU>, MODE, EPI>), dim3((unsigned)plan.tiles), dim3(256), 0, s, g);
}
// Subchannel: the 128 x 128 tile of shk_f6sub.h (SwiGLU: 128 x 64 outputs).
// Without it M, N or K off the FP6 entry's 128 ran the register-staged 64 x
// 64 tile, and SwiGLU the 256 x 64 one.
template <bool SWIGLU>
using CSub = Cfg<4, true, true, 128, SWIGLU ? 64 : 128, 128, 2, 2, SWIGLU, true, 64, false, 0>;

template <bool SWIGLU, int MODE, int EPI>
void launch_sub_edge(const DenseArgs& g, hipStream_t s) {
  using T = CSub<SWIGLU>;
  // (whole tile rows, and one more for the rows left over)
  const dim3 grid((unsigned)(((g.M + T::BM - 1) / T::BM) * ((g.N + T::BN - 1) / T::BN)));
  if (g.subchannel == 32) hipLaunchKernelGGL((f6_sub_edge_kernel<T, MODE, EPI, 1>), grid, dim3(256), 0, s, g);
  else if (g.subchannel == 64) hipLaunchKernelGGL((f6_sub_edge_kernel<T, MODE, EPI, 2>), grid, dim3(256), 0, s, g);
  else if (g.subchannel == 128) hipLaunchKernelGGL((f6_sub_edge_kernel<T, MODE, EPI, 4>), grid, dim3(256), 0, s, g);
  else hipLaunchKernelGGL((f6_sub_edge_kernel<T, MODE, EPI, 8>), grid, dim3(256), 0, s, g);
}

template <bool SWIGLU, bool SUB, int MODE, int EPI>
void launch_gemm(const DenseArgs& g, hipStream_t s) {
  if constexpr (SUB) launch_sub_edge<SWIGLU, MODE, EPI>(g, s);
  else launch_edge<SWIGLU, MODE, EPI>(g, s);
}
template <bool SWIGLU, bool SUB>
hipError_t launch_f6_edge(const DenseArgs& a, dim3, hipStream_t s) {
  F6PackArgs pa = f6_pack_args(a, 0, SWIGLU), pb = f6_pack_args(a, 1, SWIGLU);
  if (SUB) pb.swiglu_shift = 5;
  // per-channel calls interleave the two conversions, subchannel ones run A's
  // first, as the FP6 entries do
  hipError_t err = launch_f6_pack2(pa, f6_mn_major(a, 0), pb, f6_mn_major(a, 1), s, nullptr, !SUB);
  if (err != hipSuccess) return err;
  DenseArgs g = a;
  g.a = a.work;
  g.b = f6_work_b(a);
  const bool relu2 = !SWIGLU && a.epilogue == EPI_RELU2;
  constexpr int R2 = SWIGLU ? EPI_NONE : EPI_RELU2;
  if (a.out_mode == OUT_I32) launch_gemm<SWIGLU, SUB, OUT_I32, EPI_NONE>(g, s);
  else if (a.out_mode == OUT_F32)
    relu2 ? launch_gemm<SWIGLU, SUB, OUT_F32, R2>(g, s) : launch_gemm<SWIGLU, SUB, OUT_F32, EPI_NONE>(g, s);
  else
    relu2 ? launch_gemm<SWIGLU, SUB, OUT_BF16, R2>(g, s) : launch_gemm<SWIGLU, SUB, OUT_BF16, EPI_NONE>(g, s);
  return hipGetLastError();
}

// The entry's tile is its granularity; num_stages and LDS are those of the
// largest kernel it may launch.
template <bool SWIGLU, bool SUB>
Entry edge_entry(int layout, int bm) {
  constexpr int BN = SWIGLU ? 128 : 256;
  shk_kernel_desc d = desc_of<C<BN, SWIGLU>>(SHK_FAMILY_DENSE, layout, 8);
  d.block_m = bm;
  d.block_n = 64;
  d.block_k = SUB ? 64 : 32;
  d.num_stages = F6Engine<C<BN, SWIGLU>>::P;
  d.lds_bytes = F6Engine<C<BN, SWIGLU>>::LDS_BYTES + MFMA32_SCALE_BYTES;
  if (SUB) {
    d.scale_mode = SHK_SCALE_SUBCHANNEL;
    d.min_subchannel = 32;
    d.max_subchannel = 256;
    d.num_stages = F6SubEngine<CSub<SWIGLU>>::P;
    d.lds_bytes = f6_sub_lds_bytes<CSub<SWIGLU>>();
  }
  d.operand_format = SHK_OPERANDS_FP6_EDGE;
  return Entry{d, &launch_f6_edge<SWIGLU, SUB>, nullptr, nullptr, nullptr};
}

}  // namespace

void append_edge_f6(std::vector<Entry>& t, int layout) {
  for (int bm : {64, 16}) {
    t.push_back(edge_entry<false, false>(layout, bm));
    t.push_back(edge_entry<true, false>(layout, bm));
    t.push_back(edge_entry<false, true>(layout, bm));
    t.push_back(edge_entry<true, true>(layout, bm));
  }
}

}  // namespace shk
