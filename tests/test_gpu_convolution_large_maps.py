"""Convolution weight gradients over maps so large, or batches so long, that the
product kernel's narrow loaders (24-bit products, 32-bit byte offsets) do not
take them. Inputs are small integers and delta is sparse, so every summation
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


@pytest.mark.parametrize("batch,H,W,ks", [(2, 4096, 4096, 1), (2, 4096, 4096, 3), (2, 5000, 5000, 3), (3, 2, 9000001, 1)])
def test_positions_past_24_bits(dev, batch, H, W, ks):
    """2^24 and more positions an image, in the second and third image too."""
    _case(batch, 1, H, W, 1, ks, 1, ks // 2)


def test_images_past_24_bits(dev):
    """2^24 + 5 images of one position."""
    _case((1 << 24) + 5, 1, 1, 1, 1, 3, 1, 1)
