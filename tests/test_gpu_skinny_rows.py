"""The skinny entries that plan their rows (shk_table.h sk_plan): a call of M
rows runs 16-, 32- or 64-row tiles masked to M.  Every output against the CPU
oracle; the row below the output stays untouched, and the workspace of a split
K is left zero."""

from __future__ import annotations

import itertools

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
    assert kt.sk_plan(bits, sub, swiglu, m, n, k, kt.LAYOUT_CODES[layout])[0] == rows
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


def _shape(bits, sub, swiglu, layout, rows, masked, split, groups=None):
    """The least work whose plan is tiles of `rows` rows, masked or whole, with
    or without K split over workgroups."""
    code = kt.LAYOUT_CODES[layout]
    ks = [groups * sub + (32 if groups * sub % 64 else 0)] if sub else [96, 160, 544, 1056, 2080, 4128, 8192, 13632]
    shapes = sorted(itertools.product(range(16, 305, 16), (64, 192, 512, 1024, 2048, 3072, 4096, 8192), ks),
                    key=lambda s: s[0] * s[1] * s[2])
    for m, n, k in shapes:
        if bool(m % rows) != masked or kt.sk_plan(bits, sub, swiglu, m, n, k, code)[0] != rows:
            continue
        if sub or (kt._sk_splits(bits, -(-m // rows) * (n // 64), k) > 1) == split:
            return m, n, k
    raise LookupError


# every height masked and whole, with K split where a plan of the height splits it
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("rows,masked,split", [(16, False, False), (16, False, True), (32, True, False), (32, False, False),
                                               (32, True, True), (64, True, False), (64, False, False), (64, True, True)])
def test_every_height_matches_the_oracle(bits, epilogue, rows, masked, split, layout, device):
    m, n, k = _shape(bits, 0, epilogue == "swiglu", layout, rows, masked, split)
    _check(bits, layout, epilogue, 0, m, n, k, device, rows)


# one to three groups, and more than the waves of a tile take in one round (16
# rows 8 or 16 groups, 32 rows 8, SwiGLU 4): the totals carry over in group order
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("sub", [32, 64, 128, 256])
@pytest.mark.parametrize("epilogue,rows,masked,groups", [("none", 16, False, 2), ("none", 32, True, 2), ("none", 32, True, 9),
                                                         ("none", 32, False, 37), ("swiglu", 32, True, 37),
                                                         ("swiglu", 32, False, 9)])
def test_subchannel_heights_match_the_oracle(bits, sub, epilogue, rows, masked, groups, layout, device):
    m, n, k = _shape(bits, sub, epilogue == "swiglu", layout, rows, masked, False, groups)
    _check(bits, layout, epilogue, sub, m, n, k, device, rows)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k", [(64, 6720, 13632), (480, 896, 13824)])
def test_int4_64_row_tiles_with_k_split(m, n, k, layout, device):
    """64-row tiles, whole and masked, of which two workgroups share the K."""
    _check(4, layout, "none", 0, m, n, k, device, 64, splits=2)
