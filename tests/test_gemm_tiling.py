"""The tilings of matrix products (gemm_tiling.hpp), on the host: what the kernel
and its scratch take for granted."""

from __future__ import annotations

import math

import numpy as np
import pytest

from tests.tilings import OWN, SHARED, tiling

TILES = {(128, 128): 2, (128, 64): 3, (64, 128): 3, (64, 64): 4, (32, 128): 4}  # workgroups a CU


def _check(m, n, k, z, floats, wide):
    t = tiling(m, n, k, z, floats, wide)
    tiles = -(-m // t.bm) * -(-n // t.bn) * z
    slabs = -(-k // 16)
    assert (t.bm, t.bn) in TILES and (not wide or (t.bm, t.bn) == (64, 64))
    assert t.k_chunk % 16 == 0
    if t.splits > 1 or t.stream:
        assert z == 1 and k >= 128 and floats > 0
    if t.stream:
        assert t.splits == 1 and 4 <= t.stream < slabs
        rest = tiles - t.full_tiles
        assert t.full_tiles % (256 * TILES[t.bm, t.bn]) == 0 and 0 < rest < 256 * TILES[t.bm, t.bn]
        runs = -(-rest * slabs // t.stream)
        assert rest * slabs + t.stream < 2**31
        assert (runs + rest) * t.bm * t.bn <= floats  # piece (run b, tile t) has partial tile b + t
    else:
        assert t.full_tiles == 0 and 1 <= t.splits <= 1024
        if t.splits > 1:
            assert t.splits * m * n <= floats
        if k > 0:
            assert (t.splits - 1) * t.k_chunk < k <= t.splits * t.k_chunk  # no empty range, none missing


@pytest.mark.parametrize("floats", [SHARED, OWN, 1 << 20, 1, 0])
@pytest.mark.parametrize("wide", [False, True])
def test_pieces_fit_their_scratch(floats, wide):
    r = np.random.default_rng(floats + wide)
    for _ in range(4000):
        m, n = (int(math.exp(r.uniform(0, math.log(2**20)))) for _ in range(2))
        k = int(math.exp(r.uniform(0, math.log(2**31 - 1))))
        _check(m, n, k, 1, floats, wide)
        _check(m, n, min(k, 10000), int(r.integers(2, 500)), floats, wide)


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 1, 2**31), (2**31 - 1, 1, 1), (1, 2**31 - 1, 128), (46340, 46340, 46340), (5, 7, 0),
                                   (128 * 511, 128, 5000), (128 * 513, 128, 5000), (64, 64, 127), (64, 64, 128)])
def test_edges(m, n, k):
    for floats in (SHARED, OWN, 0):
        _check(m, n, k, 1, floats, False)
