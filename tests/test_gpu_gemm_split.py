"""dkz_gemm's split of fp32 operands into three bf16 values each (h + m + l).

Six of the nine products are kept; what the split cannot hold -- infinities,
NaNs, values that round to a bf16 infinity, values so small that l (or m, or h)
falls below bf16's smallest denormal -- goes through the fp32 matrix
instruction, tile by tile, and so do products with one k. Tolerance for finite results: Higham's bound for any
fp32 summation order, gamma_(k+3) * sum |a||b| (as in test_gpu_gemm), plus
k * 2^-149 for products below fp32's range. Infinities and NaNs must be where
IEEE arithmetic on the same operands puts them.
"""

from __future__ import annotations

import numpy as np
import pytest

from darknet_zig_amd import gpu
from tests.helpers import rng
from tests.test_gpu_gemm import VARIANTS, bound, layout, run_gpu
from tests.tilings import tiling

pytestmark = pytest.mark.gpu

# Tiles with 1, 16 and 17 k (no whole slab, one, one and a tail), K whole and in
# ranges; odd rows and columns.
SHAPES = {
    (3, 5, 7): "64x64 whole",
    (65, 130, 300): "64x64 ranges",
    (2049, 4100, 1): "128x64 whole",
    (2049, 4100, 16): "128x64 whole",
    (2050, 4099, 17): "128x64 whole",
    (1385, 4458, 1): "128x128 whole",
    (1385, 4458, 16): "128x128 whole",
    (1385, 4458, 17): "128x128 whole",
    (2047, 2047, 2300): "128x128 ranges",
    (2047, 2050, 1030): "128x128 streamed",
}


def product(A, B, ta=False, tb=False):
    m, k = A.shape
    n = B.shape[1]
    ga, lda, gb, ldb = layout(A, B, ta, tb)
    gc = np.full((m, n), np.nan, np.float32)
    return run_gpu(ta, tb, m, n, k, 1.0, ga, lda, gb, ldb, 0.0, gc, n)


def check(A, B, ta=False, tb=False):
    got = product(A, B, ta, tb).astype(np.float64)
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(want), np.isnan(got))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    k = A.shape[1]
    with np.errstate(all="ignore"):
        bd = bound(A, B, np.zeros_like(want, dtype=np.float32), 1.0, 0.0, k) + k * 2.0 ** -149
        bad = fin & ~(np.abs(got - want) <= bd)
    assert not bad.any(), f"{int(bad.sum())} beyond the bound"


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("ta,tb", VARIANTS)
def test_shapes(dev, ta, tb, m, n, k):
    assert tiling(m, n, k).kind == SHAPES[m, n, k]
    r = rng(m + n + k)
    check(r.normal(size=(m, k)).astype(np.float32), r.normal(size=(k, n)).astype(np.float32), ta, tb)


@pytest.mark.parametrize("m,n,k", [(20, 64, 1000), (21, 65, 1000), (20, 64, 5000), (21, 65, 5000), (7, 12, 50000), (1, 9, 50176)])
def test_k_in_ranges(dev, m, n, k):
    """16, 79 and 448 partials, one and sixteen lanes an output, in float4s and
    floats."""
    assert tiling(m, n, k).splits in (16, 79, 447, 448)
    r = rng(m + n + k)
    check(r.normal(size=(m, k)).astype(np.float32), r.normal(size=(k, n)).astype(np.float32))


@pytest.mark.parametrize("ta,tb", VARIANTS)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.float32(3.4028235e38), np.float32(3.3961e38)])
def test_values_the_split_cannot_hold(dev, ta, tb, value):
    """One such value in each operand: its row (column) carries it, every
    other tile is what it was without it. The other factors are below 1/8, so
    no sum of finite values overflows."""
    r = rng(11)
    A = r.uniform(-0.125, 0.125, (150, 70)).astype(np.float32)
    B = r.uniform(-0.125, 0.125, (70, 200)).astype(np.float32)
    A[3, 5] = value
    check(A, B, ta, tb)
    A[3, 5] = 0.0
    B[66, 140] = value  # in the tail slab
    B[9, 0] = -0.0
    check(A, B, ta, tb)


@pytest.mark.parametrize("ta,tb", VARIANTS)
@pytest.mark.parametrize("ea,eb", [(-100, 0), (-120, 20), (-120, 110), (-135, 10), (-148, 40), (-60, -60), (-75, -70), (0, -126)])
def test_tiny_operands(dev, ta, tb, ea, eb):
    """Operands scaled by 2^ea and 2^eb: each keeps fp32's relative accuracy
    (rounded to its own denormals) at every scale."""
    r = rng(7)
    A = np.ldexp(r.normal(size=(70, 50)), ea).astype(np.float32)
    B = np.ldexp(r.normal(size=(50, 90)), eb).astype(np.float32)
    check(A, B, ta, tb)


def test_rows_of_many_scales(dev):
    """Rows from 1 down to 2^-140 in one tile, zeros among them."""
    r = rng(8)
    A = r.normal(size=(128, 64))
    A = np.ldexp(A, -(np.arange(128) % 71 * 2)[:, None]).astype(np.float32)
    A[5] = 0.0
    A[7, ::3] = 0.0
    check(A, r.normal(size=(64, 64)).astype(np.float32))
    check(np.ascontiguousarray(r.normal(size=(64, 64)).astype(np.float32)), np.ascontiguousarray(A.T))


@pytest.mark.parametrize("ta,tb", VARIANTS)
@pytest.mark.parametrize("side", ["A", "B"])
def test_tiny_values_beside_normal_ones(dev, ta, tb, side):
    """One tiny value a row, of every scale from 2^-95 to 2^-149, among normal
    ones that meet zeros, so that it alone makes up the row's results."""
    r = rng(12)
    m, k, n = 165, 70, 64
    A = r.normal(size=(m, k)).astype(np.float32)
    B = np.zeros((k, n), np.float32)
    at = 37
    A[:, at] = np.ldexp(r.uniform(1, 2, m) * r.choice([-1, 1], m), -(95 + np.arange(m) % 55)).astype(np.float32)
    B[at] = np.ldexp(r.uniform(1, 2, n), 60).astype(np.float32)
    if side == "A":
        check(A, B, ta, tb)
    else:
        check(np.ascontiguousarray(B.T), np.ascontiguousarray(A.T), ta, tb)


def test_closer_to_f64_than_the_fp32_matrix_instruction(dev):
    """Rms error over K = 1 .. 4096 against the fp32 instruction's model (every
    product added with one rounding): no larger."""
    r = rng(9)
    for k in (1, 2, 5, 16, 256, 4096):
        A, B = r.normal(size=(64, k)).astype(np.float32), r.normal(size=(k, 64)).astype(np.float32)
        want = A.astype(np.float64) @ B.astype(np.float64)
        chain = np.zeros((64, 64), np.float32)
        for p in range(k):  # fma: the product exact, the sum rounded
            chain = (chain.astype(np.float64) + np.outer(A[:, p].astype(np.float64), B[p].astype(np.float64))).astype(np.float32)
        err = np.linalg.norm(product(A, B) - want)
        assert err <= np.linalg.norm(chain - want), k


@pytest.mark.parametrize("ta,tb", VARIANTS)
def test_one_k_rounds_once(dev, ta, tb):
    """An outer product is the correctly rounded one, bit for bit."""
    r = rng(10)
    A, B = r.normal(size=(130, 1)).astype(np.float32), r.normal(size=(1, 300)).astype(np.float32)
    np.testing.assert_array_equal(product(A, B, ta, tb), A * B)
