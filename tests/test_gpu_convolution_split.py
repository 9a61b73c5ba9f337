"""The convolution entry points where their product kernel's tiles, slabs and
operand loaders end: 32-row tiles, 27 k (one whole slab of 16 and a tail), K in
several ranges, windows over 32 wide (64-bit gathers), one to three positions an
image (64-bit weight-gradient loads), positions that are no multiple of four,
many images in one tile -- and infinities and NaNs, which take the fp32 matrix
instruction. References and tolerances are test_gpu_convolution's."""

from __future__ import annotations

import numpy as np
import pytest

from darknet_zig_amd import gpu
from oracle import ref
from tests import test_gpu_convolution as base
from tests.helpers import down, rng, up

pytestmark = pytest.mark.gpu

SHAPES = [
    # batch, groups, channels, height, width, filters, ksize, stride, pad
    (2, 1, 3, 33, 31, 20, 3, 1, 1),    # 27 k, a 32-row tile
    (8, 1, 3, 40, 40, 32, 3, 2, 1),    # the same, stride 2
    (1, 1, 512, 13, 13, 96, 3, 1, 1),  # one small image: K in ranges
    (2, 2, 64, 9, 9, 72, 3, 1, 1),     # two groups: K whole
    (2, 1, 2, 36, 36, 4, 33, 1, 2),    # a window of 33
    (2, 1, 4, 35, 70, 6, 34, 33, 1),   # the same with stride 33
    (2, 1, 4, 21, 19, 6, 7, 2, 3),
    (3, 1, 5, 1, 1, 4, 1, 1, 0),       # one position an image
    (7, 1, 4, 3, 1, 5, 3, 1, 1),       # three
    (9, 1, 6, 2, 2, 33, 1, 1, 0),      # four
    (300, 1, 3, 3, 3, 130, 3, 1, 1),   # fourteen images in a column tile
    (40, 1, 20, 13, 13, 33, 3, 1, 1),
    (3, 1, 140, 5, 7, 130, 1, 1, 0),   # 35 positions, ksize 1
    (1, 1, 7, 40, 50, 129, 1, 1, 0),
    (2, 1, 130, 24, 24, 128, 3, 2, 1),  # four phases of 144 positions
]


@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_forward(dev, case):
    base.test_convolution_forward(dev, case)


@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_weight_gradient(dev, case):
    base.test_convolution_weight_gradient(dev, case)


@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_data_gradient(dev, case):
    base.test_convolution_data_gradient(dev, case)


@pytest.mark.parametrize("case", [(150, 2, 6, 1, 1, 70, 1, 1, 0), (5, 1, 130, 2, 3, 65, 1, 3, 0), (700, 1, 40, 1, 1, 33, 1, 1, 0),
                                  (300, 1, 5, 1, 2, 9, 1, 1, 0), (130, 2, 6, 3, 1, 4, 3, 1, 1)], ids=str)
def test_weight_gradient_of_one_to_three_positions(dev, case):
    """One position with ksize 1 is a TN product over the images (also of an
    image larger than the positions read); the others take 64-bit quads, K in
    ranges."""
    base.test_convolution_weight_gradient(dev, case)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("case", [(2, 1, 8, 9, 9, 40, 3, 1, 1), (2, 1, 8, 8, 8, 40, 1, 1, 0)], ids=str)
def test_values_that_are_not_finite(dev, case, value):
    """One such element of the input: the outputs and weight updates it
    reaches are what IEEE arithmetic makes them, the others within the bound."""
    batch, groups, C, H, W, F, ks, s, p = case
    r = rng(3)
    x = r.uniform(-1, 1, batch * C * H * W).astype(np.float32)
    x[C * H * W + 3 * H * W + 4 * W + 5] = value
    w = r.uniform(0.1, 1, F * C * ks * ks).astype(np.float32)
    n = ref.conv_out_dim(H, ks, s, p) * ref.conv_out_dim(W, ks, s, p)
    d = r.uniform(0.1, 1, batch * F * n).astype(np.float32)
    with np.errstate(all="ignore"):
        fwd = base._reference(case, x, w, np.zeros(batch * F * n, np.float32))[:2]
        wgr = base._wgrad_reference(case, x, d, np.zeros(w.size, np.float32))
    dx, dw, dd = up(x), up(w), up(d)
    out, upd = gpu.alloc(d.size), gpu.alloc(w.size)
    gpu.convolutionForward(batch, groups, C, H, W, F, ks, s, p, dw, dx, out)
    gpu.convolutionWeightGradient(batch, groups, C, H, W, F, ks, s, p, dd, dx, upd)
    for got, (want, bd) in ((down(out, d), fwd), (down(upd, w), wgr)):
        assert np.array_equal(np.isnan(got), np.isnan(want))
        inf = np.isinf(want)
        assert np.array_equal(got[inf], want[inf].astype(np.float32))
        fin = np.isfinite(want)
        assert fin.any() and not fin.all()
        assert np.all(np.abs(got[fin] - want[fin]) <= bd[fin])
    for b in (dx, dw, dd, out, upd):
        gpu.free(b)


def test_tiny_weights_beside_normal_ones(dev):
    """Kernels whose centre tap alone meets the image (one pixel an image, the
    other taps outside it): a centre of 2^-112 to 2^-140 beside taps near 1."""
    case = (70, 1, 3, 1, 1, 29, 3, 1, 1)
    batch, groups, C, H, W, F, ks, s, p = case
    r = rng(6)
    w = r.uniform(0.5, 1, (F, C, 9)).astype(np.float32)
    w[:, :, 4] = np.ldexp(w[:, :, 4], -112 - np.arange(F)[:, None]).astype(np.float32)
    x = np.ldexp(r.uniform(0.5, 1, batch * C), 40).astype(np.float32)
    want, bd, _ = base._reference(case, x, w.ravel(), np.zeros(batch * F, np.float32))
    dx, dw, out = up(x), up(w.ravel()), gpu.alloc(batch * F)
    gpu.convolutionForward(batch, groups, C, H, W, F, ks, s, p, dw, dx, out)
    got = down(out, np.empty(batch * F, np.float32)).astype(np.float64)
    for b in (dx, dw, out):
        gpu.free(b)
    assert np.all(np.abs(got - want) <= bd)


@pytest.mark.parametrize("case", [(42, 1, 75, 31, 31, 18, 1, 1, 0), (61, 1, 3, 19, 19, 23, 1, 1, 0), (9, 1, 6, 122, 122, 46, 3, 2, 1)], ids=str)
def test_many_ranges_of_k_lose_nothing(dev, case):
    """Weight gradients whose K is cut into a hundred ranges and more, positive
    data. With u = 2^-24: the sum's one rounding leaves at most u, u / sqrt(3)
    rms; a range of 20 slabs, rounded twice a slab at partial sums that grow to
    the range's, at most sqrt(40 / 3) u / sqrt(3) rms, and a hundred independent
    ranges a tenth of that: 0.62 u together. A fp32 sum of the ranges alone would
    come to about sqrt(100 / 3) u / sqrt(3) = 3.3 u."""
    batch, groups, C, H, W, F, ks, s, p = case
    r = rng(8)
    n = ref.conv_out_dim(H, ks, s, p) * ref.conv_out_dim(W, ks, s, p)
    x = r.uniform(0.1, 1, batch * C * H * W).astype(np.float32)
    d = r.uniform(0.1, 1, batch * F * n).astype(np.float32)
    want, _ = base._wgrad_reference(case, x, d, np.zeros(F * C * ks * ks, np.float32))
    dx, dd, upd = up(x), up(d), gpu.alloc(F * C * ks * ks)
    gpu.convolutionWeightGradient(batch, groups, C, H, W, F, ks, s, p, dd, dx, upd)
    got = down(upd, np.empty(want.size, np.float32)).astype(np.float64)
    for b in (dx, dd, upd):
        gpu.free(b)
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel <= 0.62 * 2.0 ** -24, rel


@pytest.mark.parametrize("ks", [1, 3, 5])
def test_one_image_of_one_position_rounds_once(dev, ks):
    """Weight gradients that are outer products: correctly rounded."""
    r = rng(13)
    C, F = 70, 40
    x, d = r.normal(size=C).astype(np.float32), r.normal(size=F).astype(np.float32)
    dx, dd, upd = up(x), up(d), gpu.alloc(F * C * ks * ks)
    gpu.convolutionWeightGradient(1, 1, C, 1, 1, F, ks, 1, ks // 2, dd, dx, upd)
    got = down(upd, np.empty(F * C * ks * ks, np.float32)).reshape(F, C, ks, ks)
    for b in (dx, dd, upd):
        gpu.free(b)
    want = np.zeros_like(got)
    want[:, :, ks // 2, ks // 2] = np.outer(d, x)
    np.testing.assert_array_equal(got, want)
