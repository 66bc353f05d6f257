"""Group sizes that a ragged call refuses: the fp6 kernels run while the host
still checks them, so they have to be safe for any sizes, and the call raises
what it always raised, before any other error of the same call."""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import amd_strix_halo_kernels as shk  # noqa: E402
from amd_strix_halo_kernels import kernel_table as kt  # noqa: E402
from amd_strix_halo_kernels import native  # noqa: E402
from tests._util import spec_of  # noqa: E402

BIG = 2**31 - 1


def _operands(device, rows=200, k=128, n=64, groups=3, layout="nn"):
    lhs = torch.randint(0, 256, (k // 2, rows) if layout == "tn" else (rows, k // 2), dtype=torch.uint8, device=device)
    rhs = torch.randint(0, 256, (groups, k // 2, n), dtype=torch.uint8, device=device)
    return lhs, rhs


def _skinny_rows(lhs, rhs, layout, sub, rows, n, k, groups):
    return native.ragged_fwd_rows(lhs, rhs, layout=shk.GemmLayout(layout), subchannel=sub, rows=rows, cols=n,
                                  k_packed=k // 2, groups=groups)


# (scale groups, layout, rows, N, rows of the skinny tiles that run): every
# kernel of the fp6 forward, the skinny tiles' per-channel and subchannel (four
# and eight waves) and the fp6 tiles' on operands that the skinny ones refuse
_PATHS = [(None, "nn", 200, 64, 64), (None, "nn", 30, 64, 16), (None, "tn", 200, 64, 0), (None, "nn", 200, 72, 0),
          (128, "nn", 200, 64, 0), (128, "nn", 30, 64, 16), (32, "nn", 30, 64, 16), (128, "nn", 100, 64, 32),
          (32, "tn", 200, 64, 0)]


@pytest.mark.parametrize("sub,layout,rows,n,skinny", _PATHS)
@pytest.mark.parametrize("delta", ["short", "long", "far", "negative", "overflow", "wraps"])
def test_forward_refuses_bad_sizes_and_stays_whole(sub, layout, rows, n, skinny, delta, device):
    sizes = {"short": [rows // 2, rows // 4, rows - rows // 2 - rows // 4 - 1], "long": [rows // 2, rows - rows // 2, 1],
             "far": [0, rows, 5000], "negative": [rows + 50, 0, -50], "overflow": [BIG, BIG, BIG],
             "wraps": [BIG, 2, 300]}[delta]
    message = {"short": f"must equal lhs rows {rows}; got {rows - 1}", "long": f"got {rows + 1}",
               "far": f"got {rows + 5000}", "negative": "non-negative", "overflow": "got 6442450941",
               "wraps": "got 2147483949"}[delta]
    lhs, rhs = _operands(device, rows=rows, n=n, layout=layout)
    assert _skinny_rows(lhs, rhs, layout, sub, rows, n, 128, 3) == skinny
    spec = spec_of(sub)
    kw = dict(scale=spec, layout=shk.GemmLayout(layout))
    print(f"case sub={sub} layout={layout} rows={rows} n={n} sizes={sizes}", flush=True)
    for dtype in (torch.int32, torch.int64):
        gs = torch.tensor(sizes, dtype=dtype, device=device)
        with pytest.raises(ValueError, match=message):
            shk.ragged_dot_int4(lhs, rhs, gs, **kw)
        # the sizes' error comes before the scales'
        with pytest.raises(ValueError, match=message):
            shk.ragged_dot_int4(lhs, rhs, gs, a_scale=torch.ones(7, device=device), **kw)
        # a caller's output is not touched by a refused call
        out = torch.full((rows, n), 3.0, dtype=torch.bfloat16, device=device)
        with pytest.raises(ValueError, match=message):
            shk.ragged_dot_int4(lhs, rhs, gs, out=out, **kw)
        torch.cuda.synchronize()
        assert bool((out == 3.0).all())
    good = torch.tensor([rows - 10, 0, 10], device=device)
    out = torch.empty((rows, n), dtype=torch.bfloat16, device=device)
    a = shk.ragged_dot_int4(lhs, rhs, good, **kw)
    b = shk.ragged_dot_int4(lhs, rhs, good.cpu(), out=out, **kw)
    assert torch.equal(a, b)


@pytest.mark.parametrize("sub", [None, 64, 128])
@pytest.mark.parametrize("sizes,message", [([129, 0, 4], "<= logical padded K 128; got 129"), ([5, -1, 4], "non-negative"),
                                           ([BIG, 1, 1], "got 2147483647")])
def test_backward_refuses_bad_sizes_and_stays_whole(sub, sizes, message, device):
    lhs = torch.randint(0, 256, (3, 96, 64), dtype=torch.uint8, device=device)
    rhs = torch.randint(0, 256, (3, 64, 64), dtype=torch.uint8, device=device)
    family = kt.FAMILY_RAGGED_BWD
    assert kt.ragged_fp6_eligible(family, subchannel=sub, m=96, n=64, k_packed=64)  # the calls whose check is deferred
    print(f"case sub={sub} sizes={sizes}", flush=True)
    kw = dict(scale=spec_of(sub))
    gs = torch.tensor(sizes, device=device)
    with pytest.raises(ValueError, match=message):
        shk.ragged_dot_int4_bwd(lhs, rhs, gs, **kw)
    with pytest.raises(ValueError, match=message):
        shk.ragged_dot_int4_bwd(lhs, rhs, gs, b_scale=torch.ones(7, device=device), **kw)
    good = torch.tensor([128, 0, 77], device=device)
    a = shk.ragged_dot_int4_bwd(lhs, rhs, good, **kw)
    b = shk.ragged_dot_int4_bwd(lhs, rhs, good.cpu(), **kw)
    assert torch.equal(a, b)


def test_capture_refuses_sizes_on_the_device(device):
    """A captured call needs its sizes on the host; device sizes still raise."""
    lhs, rhs = _operands(device)
    gs = torch.tensor([150, 0, 50], device=device)
    shk.ragged_dot_int4(lhs, rhs, gs)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        graph.capture_begin()
        assert torch.cuda.is_current_stream_capturing()
        with pytest.raises(RuntimeError):
            shk.ragged_dot_int4(lhs, rhs, gs)
        try:
            graph.capture_end()
        except RuntimeError:
            pass
    torch.cuda.synchronize()


def test_calls_under_a_default_device(device):
    """A default device of the caller's does not reach the buffer that the
    check copies the sizes into."""
    lhs, rhs = _operands(device)
    gs = torch.tensor([150, 0, 50], device=device)
    bwd = torch.randint(0, 256, (3, 96, 64), dtype=torch.uint8, device=device)
    bwd_rhs = torch.randint(0, 256, (3, 64, 64), dtype=torch.uint8, device=device)
    bwd_gs = torch.tensor([128, 0, 77], device=device)
    want, want_bwd = shk.ragged_dot_int4(lhs, rhs, gs), shk.ragged_dot_int4_bwd(bwd, bwd_rhs, bwd_gs)
    with torch.device(device):
        assert torch.equal(shk.ragged_dot_int4(lhs, rhs, gs), want)
        assert torch.equal(shk.ragged_dot_int4_bwd(bwd, bwd_rhs, bwd_gs), want_bwd)
        with pytest.raises(ValueError, match="got 199"):
            shk.ragged_dot_int4(lhs, rhs, gs - torch.tensor([1, 0, 0]))
