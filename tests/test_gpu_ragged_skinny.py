"""The ragged forward's skinny tiles (k_ragskinny.hip), which run where groups
hold few rows: NN and NT, N a multiple of 16 and K of 32 (subchannel: of the
group), against the oracle.  Every output is bit-exact: integer sums, and for
subchannel scales the oracle's order."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import ref
from tests._util import bf16_bits, stable_seed
from tests.test_gpu_ragged import _fwd_case, _ragged_int_reference, _run_fwd_native

torch = pytest.importorskip("torch")

import amd_strix_halo_kernels as shk  # noqa: E402
from amd_strix_halo_kernels import kernel_table as kt  # noqa: E402
from amd_strix_halo_kernels import native  # noqa: E402

pytestmark = pytest.mark.gpu

# sizes at the edges of 16, 32 and 64-row tiles, empty groups at both ends,
# more groups than a wave has lanes; average rows that pick each tile height
SIZES = {
    "one": [1], "edges": [0, 16, 17, 0, 15, 1, 0], "rows32": [33, 0, 31, 32, 1], "rows64": [65, 64, 0, 63, 8],
    "skewed": [0, 0, 150, 0, 1, 0], "many": [(7 * g) % 5 for g in range(200)],
}


@pytest.mark.parametrize("layout", [shk.GemmLayout.NN, shk.GemmLayout.NT], ids=lambda l: l.value)
@pytest.mark.parametrize("sub", [None, 32, 64, 128, 256])
@pytest.mark.parametrize("name", SIZES)
def test_ragged_skinny_tiles_match_the_oracle(name, sub, layout, device):
    sizes = SIZES[name]
    # rows after the last group's: not written
    m = sum(sizes) + (1 if sub is None else sum(sizes) % 2)
    n, k = (80, 160) if sub is None else (48, 3 * sub if sub > 32 else 192)
    spec = shk.ScaleSpec(shk.ScaleMode.SUBCHANNEL, sub) if sub else shk.ScaleSpec(shk.ScaleMode.PER_CHANNEL)
    a_q, b_q, sa, sb = _fwd_case(stable_seed("ragskinny", name, sub, layout.value), m, k, n, sizes, spec)
    print(f"case ragged skinny {layout.value} S={sub} {name} m={m}", flush=True)
    want = ref.ragged_fwd_reference(a_q, b_q, np.array(sizes), sa, sb, subchannel=sub)
    rows = sum(sizes)
    picked = native.ragged_fwd_rows(1 << 20, 1 << 20, layout=layout, subchannel=sub, rows=m, cols=n, k_packed=k // 2,
                                    groups=len(sizes))
    assert picked > 0  # (freshly allocated operands are aligned)

    def run(mode):
        return _run_fwd_native(device, a_q, b_q, sizes, sa, sb, layout, kt.RAGGED_FP6_BLOCK_M, mode, fp6=True,
                               subchannel=sub)[:rows]

    assert np.array_equal(run(kt.OUT_F32).cpu().numpy(), want[:rows])
    assert np.array_equal(bf16_bits(torch, run(kt.OUT_BF16)), ref.bf16_round(want)[:rows])
    got = run(kt.OUT_I32).cpu().numpy().astype(np.int64)
    assert np.array_equal(got, _ragged_int_reference(a_q, b_q, sizes)[:rows])


@pytest.mark.parametrize("sub", [None, 64])
def test_both_ragged_paths_give_the_same_bits(sub, device):
    """The same call with lhs at an offset that the skinny tiles do not take
    (they want 16 bytes), with scales that are zero, tiny, infinite and NaN."""
    groups, rows, n, k = 5, 60, 112, 192
    gen = torch.Generator(device=device).manual_seed(11)
    sizes = torch.tensor([3, 0, 40, 16, 1], device=device)
    lhs = torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device=device, generator=gen)
    rhs = torch.randint(0, 256, (groups, k // 2, n), dtype=torch.uint8, device=device, generator=gen)
    cols = 1 if sub is None else k // sub
    sa = torch.rand((rows, cols), device=device, generator=gen).bfloat16()
    sb = torch.rand((groups, cols, n), device=device, generator=gen).bfloat16()
    sa[::7], sa[1::9], sb[:, 0, ::5] = 0.0, float("inf"), 2.0**-70
    sb[:, -1, 3::11] = float("nan")
    if sub is None:
        sa, sb = sa[:, 0].contiguous(), sb[:, 0].contiguous()
    spec = shk.ScaleSpec(shk.ScaleMode.SUBCHANNEL, sub) if sub else shk.ScaleSpec(shk.ScaleMode.PER_CHANNEL)
    moved = torch.empty(lhs.numel() + 8, dtype=torch.uint8, device=device)[8:].view_as(lhs)
    moved.copy_(lhs)
    picked = [native.ragged_fwd_rows(x, rhs, layout=shk.GemmLayout.NN, subchannel=sub, rows=rows, cols=n,
                                     k_packed=k // 2, groups=groups) for x in (lhs, moved)]
    assert picked[0] == 16 and picked[1] == 0
    for dtype in (torch.bfloat16, torch.float32):
        print(f"case ragged paths S={sub} {dtype}", flush=True)
        a = shk.ragged_dot_int4(lhs, rhs, sizes, a_scale=sa, b_scale=sb, scale=spec, output_dtype=dtype)
        b = shk.ragged_dot_int4(moved, rhs, sizes, a_scale=sa, b_scale=sb, scale=spec, output_dtype=dtype)
        bits = torch.int16 if dtype is torch.bfloat16 else torch.int32
        if dtype is torch.float32:  # a NaN's payload is not part of the result
            a, b = a.nan_to_num(nan=7.0, posinf=torch.inf, neginf=-torch.inf), \
                b.nan_to_num(nan=7.0, posinf=torch.inf, neginf=-torch.inf)
        assert torch.equal(a.view(bits), b.view(bits))
