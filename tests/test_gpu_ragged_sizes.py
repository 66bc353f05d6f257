"""Group sizes that a ragged call refuses: the fp6 kernels run while the host
still checks them, so they have to be safe for any sizes, and the call raises
what it always raised, before any other error of the same call."""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import amd_strix_halo_kernels as shk  # noqa: E402

BIG = 2**31 - 1


def _operands(device, rows=200, k=128, n=64, groups=3):
    lhs = torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device=device)
    rhs = torch.randint(0, 256, (groups, k // 2, n), dtype=torch.uint8, device=device)
    return lhs, rhs


@pytest.mark.parametrize("sub", [None, 128])
@pytest.mark.parametrize("sizes,message", [
    ([100, 50, 49], "must equal lhs rows 200; got 199"), ([100, 100, 1], "got 201"), ([0, 200, 5000], "got 5200"),
    ([250, 0, -50], "non-negative"), ([BIG, BIG, BIG], "got 6442450941"), ([BIG, 2, 300], "got 2147483949"),
])
def test_forward_refuses_bad_sizes_and_stays_whole(sub, sizes, message, device):
    lhs, rhs = _operands(device)
    spec = shk.ScaleSpec(shk.ScaleMode.SUBCHANNEL, sub) if sub else shk.ScaleSpec(shk.ScaleMode.PER_CHANNEL)
    print(f"case sub={sub} sizes={sizes}", flush=True)
    for dtype in (torch.int32, torch.int64):
        gs = torch.tensor(sizes, dtype=dtype, device=device)
        with pytest.raises(ValueError, match=message):
            shk.ragged_dot_int4(lhs, rhs, gs, scale=spec)
        # the sizes' error comes before the scales'
        with pytest.raises(ValueError, match=message):
            shk.ragged_dot_int4(lhs, rhs, gs, scale=spec, a_scale=torch.ones(7, device=device))
        # a caller's output is not touched by a refused call
        out = torch.full((200, 64), 3.0, dtype=torch.bfloat16, device=device)
        with pytest.raises(ValueError, match=message):
            shk.ragged_dot_int4(lhs, rhs, gs, scale=spec, out=out)
        torch.cuda.synchronize()
        assert bool((out == 3.0).all())
    good = torch.tensor([150, 0, 50], device=device)
    out = torch.empty((200, 64), dtype=torch.bfloat16, device=device)
    a = shk.ragged_dot_int4(lhs, rhs, good, scale=spec)
    b = shk.ragged_dot_int4(lhs, rhs, good.cpu(), scale=spec, out=out)
    assert torch.equal(a, b)


@pytest.mark.parametrize("sizes,message", [([129, 0, 4], "<= logical padded K 128; got 129"), ([5, -1, 4], "non-negative"),
                                           ([BIG, 1, 1], "got 2147483647")])
def test_backward_refuses_bad_sizes_and_stays_whole(sizes, message, device):
    lhs = torch.randint(0, 256, (3, 96, 64), dtype=torch.uint8, device=device)
    rhs = torch.randint(0, 256, (3, 64, 64), dtype=torch.uint8, device=device)
    print(f"case sizes={sizes}", flush=True)
    gs = torch.tensor(sizes, device=device)
    with pytest.raises(ValueError, match=message):
        shk.ragged_dot_int4_bwd(lhs, rhs, gs)
    with pytest.raises(ValueError, match=message):
        shk.ragged_dot_int4_bwd(lhs, rhs, gs, b_scale=torch.ones(7, device=device))
    good = torch.tensor([128, 0, 77], device=device)
    a = shk.ragged_dot_int4_bwd(lhs, rhs, good)
    b = shk.ragged_dot_int4_bwd(lhs, rhs, good.cpu())
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
