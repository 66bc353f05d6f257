"""Which tiles the fp6 ragged forward runs (k_ragskinny.hip ragged_skinny_rows):
the choice, by the library's answer, and the bound of its grid."""

from __future__ import annotations

import pytest

import amd_strix_halo_kernels as shk
from amd_strix_halo_kernels import native

P = 1 << 20


def _rows(m, n, k, groups, sub=None, layout="nn", lhs=P, rhs=P):
    return native.ragged_fwd_rows(lhs, rhs, layout=shk.GemmLayout(layout), subchannel=sub, rows=m, cols=n,
                                  k_packed=k // 2, groups=groups)


def test_rows_follow_the_average_group():
    assert [_rows(m, 1024, 2048, 64) for m in (64, 768, 1536, 4096)] == [16, 16, 32, 64]
    assert _rows(8192, 1408, 2048, 8) == 0
    assert [_rows(m, 1408, 2048, 8, 128) for m in (8, 64, 512, 1024)] == [16, 16, 32, 0]


@pytest.mark.parametrize("change", [dict(layout="tn"), dict(lhs=P + 8), dict(rhs=P + 8), dict(n=1016), dict(groups=1025)])
def test_calls_that_the_skinny_tiles_do_not_take(change):
    call = dict(m=64, n=1024, k=2048, groups=64)
    assert _rows(**call) == 16
    assert _rows(**{**call, **change}) == 0


@pytest.mark.parametrize("sub,threads,bn", [(128, 512, 16), (32, 256, 16), (None, 256, 64)])
def test_no_launch_of_2_32_work_items(sub, threads, bn):
    """Many experts with a very wide N: past the limit of a launch the fp6
    tiles, 128 columns wide, run as they did."""
    groups = rows = 1024
    k = 128
    tasks = groups + rows // 16
    widest = ((1 << 32) // threads - 2) // tasks * bn
    assert _rows(rows, widest, k, groups, sub) == 16
    assert (tasks * (widest // bn + 2) + 1) * threads >= 1 << 32
    assert _rows(rows, widest + 2 * bn, k, groups, sub) == 0
