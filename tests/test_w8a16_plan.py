"""Which block tile the W8A16 plan takes on 256 CUs (no GPU needed), at the lines of its rules: both sides
of each were timed, and a shape that measured faster on another kernel stays with it."""

from __future__ import annotations

import pytest

from turingserve_amd import _native as N


def tile(M, n, k):
    t = N.lib().ts_w8a16_plan_tile(M, n, k, 256)
    return (t >> 16, t >> 4 & 0xfff, t & 15) if t else None


@pytest.mark.parametrize("n,k,lines", [
    # wide and of few rows: 128 x 96 up to 96 rows, then 128 x 128 wide tiles, then two per CU
    (17920, 1536, {65: (128, 96, 2), 72: (128, 96, 2), 96: (128, 96, 2), 97: None, 128: None,
                   129: (128, 64, 2), 192: (128, 64, 2), 193: (128, 96, 2), 256: (128, 96, 2),
                   257: None, 560: (256, 192, 1), 1152: (256, 192, 1), 1664: None,
                   1856: (256, 192, 1)}),
    # short K: no 128 x 64 with four groups in place of 128 x 64 wide tiles, no 256 x 192 over
    # several rounds that it fills to 0.79
    (9728, 896, {97: None, 128: None, 160: None, 192: None, 193: (128, 96, 4), 320: (128, 128, 2),
                 1024: (256, 192, 1), 2048: None}),
    # four 128 x 32 wide tiles per CU stay
    (1152, 896, {896: None, 960: (64, 96, 4), 1664: None}),
    (2048, 1536, {512: None, 560: (64, 96, 4), 832: (128, 64, 4), 1152: (128, 96, 4),
                  1856: (128, 128, 2)}),
    (1536, 8960, {1024: (128, 64, 4), 1408: (128, 96, 4), 2048: (128, 128, 2)}),
])
def test_block_tile_at_the_lines(n, k, lines):
    assert {m: tile(m, n, k) for m in lines} == lines
