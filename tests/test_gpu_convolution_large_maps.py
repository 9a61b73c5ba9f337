"""Convolutions over maps so large, or batches so long, that the product kernel's
narrow loaders (24-bit products, 32-bit byte offsets) do not take them. Inputs are small integers and delta is sparse, so every summation
order is exact and the results must match bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from darknet_zig_amd import gpu
from tests.helpers import down, rng, up

pytestmark = pytest.mark.gpu


def _weight_gradient(x, d, ks, stride, pad):
    """sum over images and positions of delta x the tap's input, over delta's
    nonzero elements alone. x [B, C, H, W], d [B, F, Ho, Wo]."""
    (B, C, H, W), F = x.shape, d.shape[1]
    out = np.zeros((F, C, ks, ks))
    img, f, h, w = np.nonzero(d)
    v = d[img, f, h, w].astype(np.float64)
    for kh in range(ks):
        for kw in range(ks):
            y, z = h * stride + kh - pad, w * stride + kw - pad
            ok = (y >= 0) & (y < H) & (z >= 0) & (z < W)
            for c in range(C):
                t = v[ok] * x[img[ok], c, y[ok], z[ok]]
                out[:, c, kh, kw] = np.bincount(f[ok], weights=t, minlength=F)
    return out.astype(np.float32)


def _case(batch, channels, H, W, filters, ks, stride, pad, nonzeros=20000):
    r = rng(H + W + ks)
    ho, wo = (H + 2 * pad - ks) // stride + 1, (W + 2 * pad - ks) // stride + 1
    x = r.integers(-3, 4, (batch, channels, H, W), dtype=np.int8).astype(np.float32)
    d = np.zeros((batch, filters, ho, wo), np.float32)
    d.ravel()[r.integers(0, d.size, nonzeros)] = r.integers(1, 4, nonzeros)
    d[:, :, -1, -1] = 1.0  # the last position of each image
    want = _weight_gradient(x, d, ks, stride, pad)
    dx, dd, dw = up(x.ravel()), up(d.ravel()), gpu.alloc(want.size)
    gpu.convolutionWeightGradient(batch, 1, channels, H, W, filters, ks, stride, pad, dd, dx, dw)
    got = down(dw, want)
    for b in (dx, dd, dw):
        gpu.free(b)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("batch,H,W,ks", [(2, 4096, 4096, 1), (2, 4096, 4096, 3), (2, 5000, 5000, 3), (3, 2, 9000001, 1),
                                          (2, 9000001, 2, 3), (2, 1, 17000003, 3)])
def test_positions_past_24_bits(dev, batch, H, W, ks):
    """2^24 and more positions an image, in the second and third image too:
    bands of rows, of positions (ksize 1), and 64-bit loaders (sides past 2^24)."""
    _case(batch, 1, H, W, 1, ks, 1, ks // 2)


def test_bands_with_stride(dev):
    _case(1, 1, 9001, 9003, 1, 3, 2, 1)  # 4501 x 4502 outputs: two bands


def test_images_past_24_bits(dev):
    """2^24 + 5 images of one position."""
    _case((1 << 24) + 5, 1, 1, 1, 1, 3, 1, 1)


def _sparse_case(batch, channels, H, W, filters, ks, stride, pad, at=24):
    """Input and delta of zeros but for `at` positions of delta and the input's
    windows there: tensors of gigabytes without their host copies."""
    r = rng(batch + H + ks)
    ho, wo = (H + 2 * pad - ks) // stride + 1, (W + 2 * pad - ks) // stride + 1
    x, d = gpu.alloc(batch * channels * H * W), gpu.alloc(batch * filters * ho * wo)
    dw = gpu.alloc(filters * channels * ks * ks)
    values = {}  # the input's elements
    def at_x(i, c, y, z):
        return ((i * channels + c) * H + y) * W + z
    try:
        places = {(int(r.integers(batch)), int(r.integers(ho)), int(r.integers(wo))) for _ in range(at)}
        places |= {(0, 0, 0), (batch - 1, ho - 1, wo - 1), (batch - 1, ho // 2, wo // 2)}
        places = sorted(places)
        for i, h, w in places:
            z0, z1 = max(w * stride - pad, 0), min(w * stride - pad + ks, W)
            for c in range(channels):
                for y in range(max(h * stride - pad, 0), min(h * stride - pad + ks, H)):
                    row = np.array([values.setdefault(at_x(i, c, y, z), int(r.integers(1, 9))) for z in range(z0, z1)], np.float32)
                    gpu.push(x.offset(at_x(i, c, y, z0)), row)
        want = np.zeros((filters, channels, ks, ks))
        for i, h, w in places:
            for f in range(filters):
                v = int(r.integers(1, 9))
                gpu.push(d.offset(((i * filters + f) * ho + h) * wo + w), np.array([v], np.float32))
                for c in range(channels):
                    for kh in range(ks):
                        for kw in range(ks):
                            y, z = h * stride + kh - pad, w * stride + kw - pad
                            if 0 <= y < H and 0 <= z < W:
                                want[f, c, kh, kw] += v * values[at_x(i, c, y, z)]
        gpu.convolutionWeightGradient(batch, 1, channels, H, W, filters, ks, stride, pad, d, x, dw)
        np.testing.assert_array_equal(down(dw, want.astype(np.float32)), want)
    finally:
        for b in (x, d, dw):
            gpu.free(b)


@pytest.mark.parametrize("case", [
    # batch, channels, height, width, filters, ksize, stride, pad
    (5, 8, 4000, 4000, 1, 3, 1, 1),     # 2.4 GiB of input: four images a product, then one
    (3, 2, 4000, 4000, 16, 1, 1, 0),    # 2.9 GiB of delta: two images, then one
    (40, 8, 1801, 1999, 2, 3, 2, 1),    # 4.3 GiB of input, odd maps: 18, 18 and 4 images
    (1, 40, 3840, 3840, 3, 3, 1, 1),    # an image past 2^31 bytes: 64-bit addresses, K in ranges
    (2, 1, 4095, 4097, 33, 1, 1, 0),    # the same in delta
], ids=str)
def test_batches_past_2_gib(dev, case):
    _sparse_case(*case)


def test_the_longest_map(dev):
    """2^31 - 1 positions: rounded up to a multiple of four, 2^31."""
    _sparse_case(1, 1, 1, 2**31 - 1, 1, 1, 1, 0)


def test_forward_with_padding_past_2_gib(dev):
    """An image of 0.8 GB and padding larger than the window: from a window's
    first tap at (0, 0) the image's last rows lie past 2^31 bytes."""
    H, W, ks, stride, pad = 1000, 200000, 3, 16, 1700
    ho, wo = (H + 2 * pad - ks) // stride + 1, (W + 2 * pad - ks) // stride + 1
    r = rng(3)
    w = r.integers(1, 9, (ks, ks)).astype(np.float32)
    want = np.zeros((ho, wo), np.float32)
    x, dw, out = gpu.alloc(H * W), up(w.ravel()), gpu.alloc(ho * wo)
    try:
        taps = {(int(h), int(q), int(kh), int(kw)) for h, q, kh, kw in
                zip(r.integers(107, 168, 60), r.integers(107, 12606, 60), r.integers(0, ks, 60), r.integers(0, ks, 60))}
        placed = {}
        for h, q, kh, kw in taps | {(168, 12606, 0, 0), (168, 12605, 1, 2)}:
            y, z = h * stride + kh - pad, q * stride + kw - pad
            if 0 <= y < H and 0 <= z < W:
                placed[y, z] = (h, q, kh, kw, float(r.integers(1, 9)))
        assert max(y for y, _ in placed) > 980
        for (y, z), (h, q, kh, kw, v) in placed.items():  # strides past the window: one output each
            gpu.push(x.offset(y * W + z), np.array([v], np.float32))
            want[h, q] += v * w[kh, kw]
        gpu.convolutionForward(1, 1, 1, H, W, 1, ks, stride, pad, dw, x, out)
        np.testing.assert_array_equal(down(out, want), want)
    finally:
        for b in (x, dw, out):
            gpu.free(b)
