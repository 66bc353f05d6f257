"""FP6_EDGE entries (k_f6edge.hip): the fp6 tiles on shapes that are no multiple
of them, against the CPU oracle and against the skinny tiles, which read the
same operands without converting them.

int32 sums are whole numbers and equal; per-channel bf16 results scale the
same integers in the same order and equal bit for bit; SwiGLU goes through
exp and stays within 2 bf16 ulp of the oracle and one fp32 ulp of the skinny
tiles."""

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


def _kernel(fmt, layout, epilogue, sub, m):
    """The tallest entry of an operand format that divides M."""
    fits = [k for k in shk.default_registry.all() if kt.TABLE[k.table_index].operand_format == fmt
            and k.a_dtype is shk.OperandDType.INT4 and k.layout.value == layout and k.epilogue.value == epilogue
            and k.scale == spec_of(sub) and k.tile.split_k == 1 and k.schedule is shk.KernelSchedule.STANDARD
            and m % k.tile.block_m == 0]
    return max(fits, key=lambda k: k.tile.block_m)


def _operands(case, device):
    a_q, b_q, a_arg, b_arg, sa, sb = case
    return tuple(to_dev(torch, x, device) for x in (a_arg, b_arg, sa, sb))


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("epilogue", ["none", "relu2", "swiglu"])
@pytest.mark.parametrize("m,n,k", [(16, 64, 32), (48, 192, 96), (144, 320, 160), (272, 64, 416), (400, 576, 128)])
def test_edges_of_the_tiles_match_the_oracle(layout, epilogue, m, n, k, device):
    """M, N and K past, below and at the tiles' multiples (128 and 256 rows
    and columns, 128-K stages), bf16, fp32 and raw int32 outputs."""
    case = dense_case(stable_seed("edge", layout, epilogue, m, n, k), bits=4, layout=layout, m=m, n=n, k=k,
                      subchannel=None, swiglu=epilogue == "swiglu")
    kernel = _kernel(kt.OPERANDS_FP6_EDGE, layout, epilogue, None, m)
    print(f"case {kernel.kernel_id} shape=({m},{n},{k})", flush=True)
    a, b, sa, sb = _operands(case, device)
    out = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=device)
    native.launch_generated_kernel(a, b, kernel=kernel, a_scale=sa, b_scale=sb, c=out[:m])
    raw = native.launch_generated_kernel_i32(a, b, kernel=kernel, a_scale=sa, b_scale=sb)
    torch.cuda.synchronize()
    assert bool((out[m] == 7.0).all()), "rows past M written"
    assert np.array_equal(raw.cpu().numpy(), ref.int_matmul(case[0], case[1]))
    want = ref.reference_gemm_bf16(case[2], case[3], bits=4, layout=layout, a_scale=case[4], b_scale=case[5],
                                   subchannel=None, epilogue=epilogue)
    got = bf16_bits(torch, out[:m])
    assert max_ulp(got, want) <= 2 if epilogue == "swiglu" else np.array_equal(got, want)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("epilogue", ["none", "relu2", "swiglu"])
@pytest.mark.parametrize("sub", [32, 64, 128, 256])
@pytest.mark.parametrize("m,n,groups", [(16, 64, 1), (48, 192, 3), (80, 128, 2), (192, 192, 5), (240, 320, 6), (272, 128, 11)])
def test_subchannel_edges_match_the_oracle(layout, epilogue, sub, m, n, groups, device):
    """The subchannel tile at its edges: one to eleven groups (odd stage
    counts, K no multiple of 128), scales over three decades, every output."""
    k = -(-groups * sub // 64) * 64
    case = dense_case(stable_seed("edge-sub", layout, epilogue, sub, m, n, k), bits=4, layout=layout, m=m, n=n, k=k,
                      subchannel=sub, swiglu=epilogue == "swiglu", scale_lo=1e-4, scale_hi=0.1)
    kernel = _kernel(kt.OPERANDS_FP6_EDGE, layout, epilogue, sub, m)
    print(f"case {kernel.kernel_id} shape=({m},{n},{k})", flush=True)
    a, b, sa, sb = _operands(case, device)
    out = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=device)
    native.launch_generated_kernel(a, b, kernel=kernel, a_scale=sa, b_scale=sb, c=out[:m])
    raw = native.launch_generated_kernel_i32(a, b, kernel=kernel, a_scale=sa, b_scale=sb)
    torch.cuda.synchronize()
    assert bool((out[m] == 7.0).all()), "rows past M written"
    assert np.array_equal(raw.cpu().numpy(), ref.int_matmul(case[0], case[1]))
    want = ref.reference_gemm_bf16(case[2], case[3], bits=4, layout=layout, a_scale=case[4], b_scale=case[5],
                                   subchannel=sub, epilogue=epilogue)
    got = bf16_bits(torch, out[:m])
    assert max_ulp(got, want) <= 2 if epilogue == "swiglu" else np.array_equal(got, want)


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("sub", [32, 64, 128, 256])
def test_subchannel_edges_with_special_scales(sub, epilogue, device):
    """Scales outside the fast fold's range (subnormal, huge, infinite, NaN,
    signed zeros): the reference's order, NaN canonical."""
    m, n, k = 80, 128, 512
    case = list(dense_case(stable_seed("edge-special", sub, epilogue), bits=4, layout="nn", m=m, n=n, k=k,
                           subchannel=sub, swiglu=epilogue == "swiglu"))
    r = ref.rng(stable_seed("edge-special-scales", sub))
    special = np.array([0x0001, 0x0080, 0x7F7F, 0x7F80, 0xFF80, 0x7FC1, 0x0000, 0x8000, 0x2000, 0xBF80], np.uint16)
    for i in (4, 5):
        flat = case[i].reshape(-1)
        flat[::7] = special[r.integers(0, special.size, flat[::7].size)]
    kernel = _kernel(kt.OPERANDS_FP6_EDGE, "nn", epilogue, sub, m)
    a, b, sa, sb = _operands(case, device)
    got = bf16_bits(torch, shk.explicit_mm(a, b, kernel=kernel, a_scale=sa, b_scale=sb))
    with np.errstate(all="ignore"):
        want = ref.reference_gemm_bf16(case[2], case[3], bits=4, layout="nn", a_scale=case[4], b_scale=case[5],
                                       subchannel=sub, epilogue=epilogue)
    nan = (want & 0x7FFF) > 0x7F80
    assert np.array_equal(got[nan], want[nan])
    assert max_ulp(got[~nan], want[~nan]) <= 2 if epilogue == "swiglu" else np.array_equal(got, want)


# (epilogue, m, n, k): 128 x 128 tiles in two-slot rings (720 of them); all
# half-height (144 x 32704: 256 tiles of 128 rows), a whole round of large
# tiles then half-height ones (plain: 257 tiles; SwiGLU: 2 x 130), whole
# rounds only (SwiGLU 512 x 16448: 258 tiles, 2 x 129, 4 x 1 half-height)
_PLANS = [("none", 400, 23040, 32), ("none", 144, 32704, 2848), ("none", 144, 65728, 4128), ("swiglu", 272, 16576, 96),
          ("swiglu", 512, 16448, 160), ("swiglu", 1040, 8256, 64)]


@pytest.mark.parametrize("epilogue,m,n,k", _PLANS)
def test_every_tile_split_equals_the_skinny_tiles(epilogue, m, n, k, device):
    case = dense_case(stable_seed("edge-plan", epilogue, m, n, k), bits=4, layout="nt", m=m, n=n, k=k, subchannel=None,
                      swiglu=epilogue == "swiglu")
    a, b, sa, sb = _operands(case, device)
    edge, skinny = (_kernel(f, "nt", epilogue, None, m) for f in (kt.OPERANDS_FP6_EDGE, kt.OPERANDS_STREAM))
    print(f"case {edge.kernel_id} shape=({m},{n},{k})", flush=True)
    outs = [shk.explicit_mm(a, b, kernel=x, a_scale=sa, b_scale=sb) for x in (edge, skinny)]
    raws = [native.launch_generated_kernel_i32(a, b, kernel=x, a_scale=sa, b_scale=sb) for x in (edge, skinny)]
    torch.cuda.synchronize()
    assert torch.equal(raws[0], raws[1])
    got, want = (bf16_bits(torch, o) for o in outs)
    assert max_ulp(got, want) <= 2 if epilogue == "swiglu" else np.array_equal(got, want)


@pytest.mark.parametrize("layout", ["nn", "tn"])
@pytest.mark.parametrize("m,n,k,sub", [(320, 1024, 640, 128), (1344, 192, 576, 64), (320, 64, 256, 32)])
def test_calls_with_operands_at_8_bytes(m, n, k, sub, layout, device):
    """An MN-major operand that starts 8 bytes past a 16-byte boundary, as a
    view into a larger buffer may: the 64 x 64 tile's calls take it, with the
    bits of the aligned call."""
    case = dense_case(stable_seed("edge-8", m, n, k, layout), bits=4, layout=layout, m=m, n=n, k=k, subchannel=sub,
                      swiglu=False)
    a, b, sa, sb = _operands(case, device)

    def moved(t):
        buf = torch.empty(t.numel() + 16, dtype=t.dtype, device=device)
        view = buf[8:8 + t.numel()].view(t.shape)
        view.copy_(t)
        assert view.data_ptr() % 16 == 8
        return view

    kw = dict(a_scale=sa, b_scale=sb, layout=shk.GemmLayout(layout), scale=spec_of(sub))
    want = shk.mm(a, b, **kw)
    assert torch.equal(shk.mm(a, moved(b), **kw), want)
    if layout == "tn":
        assert torch.equal(shk.mm(moved(a), moved(b), **kw), want)
    else:
        with pytest.raises(RuntimeError, match="16-byte aligned A"):
            shk.mm(moved(a), b, **kw)


@pytest.mark.parametrize("mode", [kt.OUT_BF16, kt.OUT_F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("sub", [None, 32, 64, 128, 256])
def test_swiglu_is_as_precise_as_the_skinny_tiles(sub, mode, device):
    """Edge and skinny tiles share shapes, so a call must not lose precision by
    which of them it runs: the same scaled sums, gates of both signs up to some
    hundred.  Both quotients round correctly but where the edge tile's last
    rounding is a near tie (4 gates in 10^7): the fp32 results differ by one
    ulp there, and up times them may by one more."""
    m, n, k = 208, 192, 768
    case = dense_case(stable_seed("edge-swiglu", sub, mode), bits=4, layout="nn", m=m, n=n, k=k, subchannel=sub,
                      swiglu=True, scale_lo=0.02, scale_hi=0.2)
    a, b, sa, sb = _operands(case, device)
    lib = native.load_dispatch_library()
    outs = []
    for fmt in (kt.OPERANDS_FP6_EDGE, kt.OPERANDS_STREAM):
        kernel = _kernel(fmt, "nn", "swiglu", sub, m)
        out = torch.zeros((m, n), dtype=torch.bfloat16 if mode == kt.OUT_BF16 else torch.float32, device=device)
        nbytes = native.gemm_workspace_bytes(kernel, m, n, k)
        work = torch.zeros(max(nbytes, 16), dtype=torch.uint8, device=device)
        rc = lib.amd_strix_halo_kernels_launch_gemm_ws(
            kernel.table_index, 0, torch.cuda.current_stream().cuda_stream, a.data_ptr(), b.data_ptr(), sa.data_ptr(),
            sb.data_ptr(), out.data_ptr(), m, n, k, sub or 0, kt.EPILOGUE_SWIGLU, mode, work.data_ptr(), nbytes)
        torch.cuda.synchronize()
        assert rc == 0, lib.amd_strix_halo_kernels_last_error()
        outs.append(out)
    assert float(outs[0].float().abs().max()) > 100.0
    if mode == kt.OUT_BF16:
        assert torch.equal(outs[0], outs[1])
    else:
        ulps = (outs[0].view(torch.int32) - outs[1].view(torch.int32)).abs()
        assert int(ulps.max()) <= 2 and float((ulps > 0).float().mean()) <= 1e-4


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
def test_edge_entry_without_a_workspace_runs_the_packed_entry(epilogue, device):
    """A caller of the C ABI that has no workspace, or whose converted
    operands do not fit the no-allocation scratch, is served all the same."""
    m, n, k = 48, 192, 96
    swiglu = epilogue == "swiglu"
    case = dense_case(stable_seed("edge-nows", epilogue), bits=4, layout="nn", m=m, n=n, k=k, subchannel=None,
                      swiglu=swiglu)
    a, b, sa, sb = _operands(case, device)
    kernel = _kernel(kt.OPERANDS_FP6_EDGE, "nn", epilogue, None, m)
    want = bf16_bits(torch, shk.explicit_mm(a, b, kernel=kernel, a_scale=sa, b_scale=sb))
    lib = native.load_dispatch_library()
    epi = kt.EPILOGUE_SWIGLU if swiglu else kt.EPILOGUE_NONE
    for launch in (lib.amd_strix_halo_kernels_launch_gemm, lib.amd_strix_halo_kernels_launch_gemm_noalloc):
        out = torch.zeros((m, n), dtype=torch.bfloat16, device=device)
        rc = launch(kernel.table_index, 0, torch.cuda.current_stream().cuda_stream, a.data_ptr(), b.data_ptr(),
                    sa.data_ptr(), sb.data_ptr(), out.data_ptr(), m, n, k, 0, epi, kt.OUT_BF16)
        torch.cuda.synchronize()
        assert rc == 0, lib.amd_strix_halo_kernels_last_error()
        got = bf16_bits(torch, out)
        assert max_ulp(got, want) <= 2 if swiglu else np.array_equal(got, want)
    # 3/4 byte a value of 16 x 16384 and 16384 x 16384: more than the scratch
    m, n, k = 16, 16384, 16384
    assert kt.TABLE[kernel.table_index].workspace_bytes(m, n, k) > kt.NOALLOC_SCRATCH_BYTES
    a = torch.zeros((m, k // 2), dtype=torch.uint8, device=device)
    b = torch.zeros((k // 2, 2 * n if swiglu else n), dtype=torch.uint8, device=device)
    ones = torch.ones(2 * n, dtype=torch.bfloat16, device=device)
    out = torch.full((m, n), 3.0, dtype=torch.bfloat16, device=device)
    rc = lib.amd_strix_halo_kernels_launch_gemm_noalloc(kernel.table_index, 0, torch.cuda.current_stream().cuda_stream,
                                                        a.data_ptr(), b.data_ptr(), ones.data_ptr(), ones.data_ptr(),
                                                        out.data_ptr(), m, n, k, 0, epi, kt.OUT_BF16)
    torch.cuda.synchronize()
    assert rc == 0 and not bool(out.any())
