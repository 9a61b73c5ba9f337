"""The fused batch-norm passes over rows that are no whole float4s
(batchnorm_ragged.hip), at the edges of their workgroup sizes and of the choice
between one launch, two passes and the per-op sequence. References and
tolerances are test_gpu_batchnorm_fused's: statistics by the reduction rule,
everything else bit for bit given them."""

from __future__ import annotations

import numpy as np
import pytest

from darknet_zig_amd import gpu
from darknet_zig_amd.activations import Activation
from tests.helpers import down, normal, rng, uniform, up
from tests.test_gpu_batchnorm_fused import _backward_case, _forward_case

pytestmark = pytest.mark.gpu

SHAPES = [
    # batch, filters, spatial
    (1, 3, 5),         # a channel of five
    (341, 3, 3), (342, 5, 3),        # 1023 and 1026 elements: 256 threads, then 1024
    (1, 7, 4095), (1, 2, 4097),      # 4 floats a lane of 1024 threads, then 12
    (17, 5, 723), (4, 3, 3073),      # 12291 and 12292: past 12 (24 of 512)
    (7, 2, 4681), (3, 2, 10923),     # 32767 and 32769: past 32
    (5, 3, 13107), (1, 3, 65537),    # 65535 and 65537: one launch, then two passes (a split channel)
    (2, 300, 33001),                 # two passes, a workgroup a channel, n % 4 == 0
    (1, 129, 66001),                 # ... n % 4 == 1
    (4000, 17, 17),                  # two passes, 242 rows in a tile
    (64, 1024, 169),                 # 11 M elements: the forward in two passes
    (4096, 129, 1), (2048, 300, 1),  # single-element rows in one launch, and as the per-op sequence
    (40000, 2, 3),                   # three-element rows, a channel past one workgroup: the per-op sequence
]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward(dev, shape):
    _forward_case(shape, Activation.leaky, True, inplace=True, seed=sum(shape))


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_inference(dev, shape):
    _forward_case(shape, Activation.linear, False, inplace=False, seed=sum(shape) + 1)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward(dev, shape):
    _backward_case(shape, Activation.leaky, sum(shape) + 2)


@pytest.mark.parametrize("act", list(Activation), ids=lambda a: a.name)
def test_every_activation(dev, act):
    for shape in ((3, 5, 49), (2, 3, 40001)):
        _forward_case(shape, act, True, inplace=True, seed=int(act))
        _forward_case(shape, act, False, inplace=True, seed=int(act) + 20)
        _backward_case(shape, act, int(act) + 40)


@pytest.mark.parametrize("shape", [(3, 5, 16), (4, 3, 17000)], ids=str)
def test_misaligned_tensors_match_aligned_ones(dev, shape):
    """Views that start one element into a buffer: one launch, and (a channel
    past 65536 elements) the per-op sequence. Same statistics to the reduction
    rule, so element results agree to their rounding."""
    B, F, S = shape
    n = B * F * S
    r = rng(4)
    x = normal(r, n, 0.3, 1.0)
    s, b, rm, rv = uniform(r, F, 0.5, 1.5), normal(r, F, 0, 0.1), normal(r, F), uniform(r, F, 0.5, 1.5)
    out = []
    for shift in (0, 1):
        src, o, xc, xn = (up(np.concatenate([np.zeros(shift, np.float32), x if i == 0 else np.zeros(n, np.float32)]))
                          for i in range(4))
        st = [up(np.zeros(F, np.float32)) for _ in range(2)] + [up(rm), up(rv), up(s), up(b)]
        gpu.batchnormForward(B, F, S, Activation.leaky, True, *(t.offset(shift) for t in (src, o, xc, xn)), *st)
        out.append([down(t.offset(shift), x) for t in (o, xc, xn)])
        for t in (src, o, xc, xn, *st):
            gpu.free(t)
    np.testing.assert_array_equal(out[0][1], out[1][1])
    for a, c in ((out[0][0], out[1][0]), (out[0][2], out[1][2])):
        np.testing.assert_allclose(c, a, rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("at", [0, 30])
def test_values_that_are_not_finite(dev, value, at):
    """One in a channel, first or later: the per-op formulas in f64 say where
    mean, variance and outputs are infinite or NaN; other channels keep their
    values."""
    B, F, S = 3, 4, 49
    r = rng(5)
    x = normal(r, B * F * S, 0.3, 1.0).reshape(B, F, S)
    x[0, 1, at] = value
    one, zero = np.ones(F, np.float32), np.zeros(F, np.float32)
    d = [up(x.ravel()), gpu.alloc(x.size), gpu.alloc(x.size), gpu.alloc(x.size), *(up(zero) for _ in range(4)), up(one), up(zero)]
    gpu.batchnormForward(B, F, S, Activation.linear, True, *d)
    out, m, v = down(d[1], x).reshape(x.shape), down(d[4], one), down(d[5], one)
    with np.errstate(all="ignore"):
        want = x.astype(np.float64).mean(axis=(0, 2))
    assert np.array_equal(np.isnan(m), np.isnan(want)) and (np.isnan(value) or m[1] == value)
    assert np.isnan(v[1]) and np.isfinite(v[[0, 2, 3]]).all()
    assert np.isnan(out[:, 1]).all() and np.isfinite(out[:, [0, 2, 3]]).all()
    for t in d:
        gpu.free(t)
