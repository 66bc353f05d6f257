"""The skinny entries that plan their rows (shk_table.h sk_plan): a call of M
rows runs 16-, 32- or 64-row tiles masked to M.  Every output against the CPU
oracle; the row below the output stays untouched, and the workspace of a split
K is left zero."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import ref
from tests._util import bf16_bits, dense_case, max_ulp, spec_of, stable_seed, to_dev

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import amd_strix_halo_kernels as shk  # noqa: E402
from amd_strix_halo_kernels import kernel_table as kt  # noqa: E402
from amd_strix_halo_kernels import native  # noqa: E402


def _check(bits, layout, epilogue, sub, m, n, k, device, rows, splits=None):
    swiglu = epilogue == "swiglu"
    assert kt.sk_plan(bits, sub, swiglu, m, n, k)[0] == rows
    a_q, b_q, a_arg, b_arg, sa, sb = dense_case(stable_seed("rows", bits, layout, epilogue, sub, m, n, k), bits=bits,
                                                layout=layout, m=m, n=n, k=k, subchannel=sub or None, swiglu=swiglu)
    a, b, ta, tb = (to_dev(torch, x, device) for x in (a_arg, b_arg, sa, sb))
    kernel = next(x for x in shk.default_registry.all() if kt.TABLE[x.table_index].plans_rows
                  and x.scale == spec_of(sub) and x.epilogue.value == epilogue and x.layout.value == layout
                  and kt.TABLE[x.table_index].dtype_bits == bits)
    assert splits is None or kt.sk_split_count(kt.TABLE[kernel.table_index], m, n, k) == splits
    print(f"case {kernel.kernel_id} shape=({m},{n},{k}) rows={rows}", flush=True)
    out = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=device)
    for _ in range(2):  # a split launch leaves its workspace zero for the next
        native.launch_generated_kernel(a, b, kernel=kernel, a_scale=ta, b_scale=tb, c=out[:m])
    raw = native.launch_generated_kernel_i32(a, b, kernel=kernel, a_scale=ta, b_scale=tb)
    torch.cuda.synchronize()
    assert bool((out[m] == 7.0).all()), "rows past M written"
    work = native._SPLIT_WORKSPACES.get((device.index or 0, torch.cuda.current_stream(device).cuda_stream))
    assert work is None or int(work.count_nonzero()) == 0
    assert np.array_equal(raw.cpu().numpy(), ref.int_matmul(a_q, b_q))
    want = ref.reference_gemm_bf16(a_arg, b_arg, bits=bits, layout=layout, a_scale=sa, b_scale=sb,
                                   subchannel=sub or None, epilogue=epilogue)
    got = bf16_bits(torch, out[:m])
    assert max_ulp(got, want) <= 2 if swiglu else np.array_equal(got, want)


# (bits, epilogue, rows, m, n, k): masked and whole tiles of each height,
# with and without K split over workgroups
_PLANS = [
    (4, "none", 64, 112, 8192, 2080), (4, "none", 64, 192, 8192, 2080), (4, "none", 32, 48, 512, 96),
    (4, "none", 32, 144, 512, 8192), (8, "none", 64, 112, 8192, 1024), (8, "none", 32, 144, 512, 8192),
    (8, "none", 32, 112, 4096, 96), (8, "none", 64, 272, 512, 8192), (4, "swiglu", 64, 112, 8192, 96),
    (4, "swiglu", 16, 48, 512, 2080), (8, "swiglu", 64, 272, 2048, 96), (8, "swiglu", 64, 272, 512, 8192),
    (8, "swiglu", 32, 48, 512, 96), (8, "swiglu", 32, 48, 2048, 8192),
]


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("bits,epilogue,rows,m,n,k", _PLANS)
def test_every_height_matches_the_oracle(bits, epilogue, rows, m, n, k, layout, device):
    _check(bits, layout, epilogue, 0, m, n, k, device, rows)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("sub", [32, 64, 128, 256])
@pytest.mark.parametrize("epilogue,m,rows", [("none", 48, 32), ("none", 64, 32), ("swiglu", 48, 32), ("none", 32, 16)])
def test_subchannel_32_row_tiles_match_the_oracle(bits, sub, epilogue, m, rows, layout, device):
    """32-row tiles where they make fewer rounds of workgroups (N = 4096)."""
    _check(bits, layout, epilogue, sub, m, 4096 if rows == 32 else 192, (2 if sub > 64 else 5) * sub // 64 * 64 or 64,
           device, rows)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k", [(64, 6720, 13632), (480, 896, 13824)])
def test_int4_64_row_tiles_with_k_split(m, n, k, layout, device):
    """64-row tiles, whole and masked, of which two workgroups share the K."""
    _check(4, layout, "none", 0, m, n, k, device, 64, splits=2)


@pytest.mark.parametrize("layout", ["nn", "nt"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("sub", [32, 64, 128, 256])
@pytest.mark.parametrize("epilogue,m,groups", [("none", 48, 9), ("none", 64, 37), ("swiglu", 48, 37), ("swiglu", 64, 9)])
def test_subchannel_32_row_tiles_over_several_rounds(bits, sub, epilogue, m, groups, layout, device):
    """More scale groups than the waves of a 32-row tile take in one round (8,
    SwiGLU 4): the totals carry over, in group order."""
    k = -(-groups * sub // 64) * 64
    _check(bits, layout, epilogue, sub, m, 3072, k, device, 32)
