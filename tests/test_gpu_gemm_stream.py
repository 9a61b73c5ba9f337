"""Products whose last tiles are streamed: tiles that fill no whole round of the
chip have their slabs of K laid end to end and cut into equal runs, so a run may
end inside a tile and a tile's sum is that of two to a few dozen pieces. Shapes
with and without whole rounds before the streamed tiles, of 128x128, 64x64 and
32x128 tiles, with partial tiles at both edges and K that is no whole slab; C in
float4s and not. Tolerances are Higham's bound for any fp32 summation order, as
in test_gpu_gemm and test_gpu_convolution."""

from __future__ import annotations

import numpy as np
import pytest

from tests import test_gpu_convolution as base
from tests.helpers import rng
from tests.test_gpu_gemm import VARIANTS
from tests.test_gpu_gemm_split import check
from tests.tilings import OWN, SHARED, tiling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,kind", [
    (1652, 2625, 823, "128x128 streamed"),               # 273 tiles, 28 slabs a run of tiles of 52
    (2403, 3416, 164, "128x128 rounds, then streamed"),  # 512 tiles, then one streamed in runs of four slabs
    (802, 4997, 305, "64x64 rounds, then streamed"),     # 1024 tiles first
    (1281, 3146, 313, "32x128 rounds, then streamed"),   # 1024 tiles first
])
@pytest.mark.parametrize("ta,tb", VARIANTS)
def test_gemm(dev, ta, tb, m, n, k, kind):
    assert tiling(m, n, k).kind == kind
    r = rng(m + n + k)
    check(r.normal(size=(m, k)).astype(np.float32), r.normal(size=(k, n)).astype(np.float32), ta, tb)


def test_gemm_with_an_infinity(dev):
    """In a piece that starts inside a tile: only its row is not finite."""
    r = rng(7)
    A = r.uniform(0.1, 1, (1652, 823)).astype(np.float32)
    B = r.uniform(0.1, 1, (823, 2625)).astype(np.float32)
    A[900, 700] = np.inf
    check(A, B)


@pytest.mark.parametrize("case", [(39, 1, 263, 13, 13, 153, 3, 1, 1), (37, 1, 156, 14, 14, 158, 3, 1, 1)], ids=str)
def test_forward(dev, case):
    b, _, c, h, w, f, ks, _, _ = case
    assert "streamed" in tiling(f, b * h * w, c * ks * ks, floats=OWN).kind
    base.test_convolution_forward(dev, case)


@pytest.mark.parametrize("case", [(21, 1, 254, 13, 13, 366, 3, 1, 1), (39, 1, 300, 14, 14, 133, 3, 1, 1)], ids=str)
def test_weight_gradient(dev, case):
    b, _, c, h, w, f, ks, _, _ = case
    assert "streamed" in tiling(f, c * ks * ks, b * ((h * w + 3) // 4 * 4)).kind
    base.test_convolution_weight_gradient(dev, case)


@pytest.mark.parametrize("case", [(32, 1, 134, 13, 13, 360, 3, 1, 1), (37, 1, 133, 14, 14, 182, 3, 1, 1)], ids=str)
def test_data_gradient(dev, case):
    b, _, c, h, w, f, ks, _, _ = case  # the partials lie behind the flipped weights
    assert "streamed" in tiling(c, b * h * w, f * ks * ks, floats=SHARED - (f * c * ks * ks + 63) // 64 * 64).kind
    base.test_convolution_data_gradient(dev, case)
