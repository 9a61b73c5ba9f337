"""Convolution forwards and 1x1 data gradients on several streams and in captured
graphs: calls of these two may overlap on any streams, and give the same results
on all of them -- on the null stream, where pieces of a product go through a
scratch block and a reduction, and on others, where a workgroup takes all of a
tile's pieces itself. The sums of the pieces are f64 ones on both, of integers
here, so the results must match bit for bit."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from darknet_zig_amd import _lib, gpu
from oracle import ref
from tests.helpers import down, rng, up
from tests.tilings import OWN, tiling
from tests.test_gpu_streams_graphs import Hip, quiet  # noqa: F401  (quiet: a fixture)

pytestmark = pytest.mark.gpu

FORWARDS = {
    # batch, groups, channels, height, width, filters, ksize, stride, pad: the product's tiles
    (1, 1, 64, 52, 52, 128, 3, 1, 1): "64x64 ranges",
    (1, 1, 512, 13, 13, 96, 3, 1, 1): "64x64 ranges",
    (1, 1, 512, 7, 7, 10, 1, 1, 0): "64x64 ranges",
    (7, 1, 195, 32, 19, 17, 1, 1, 0): "32x128 ranges",
    (10, 1, 50, 31, 36, 34, 3, 1, 1): "64x128 ranges",
    (8, 1, 80, 29, 26, 97, 3, 1, 1): "128x64 ranges",
    (39, 1, 88, 6, 48, 68, 3, 1, 1): "128x128 ranges",
    (39, 1, 263, 13, 13, 153, 3, 1, 1): "32x128 streamed",
    (53, 1, 38, 58, 44, 18, 3, 1, 1): "32x128 rounds, then streamed",
    (15, 1, 126, 41, 18, 165, 3, 1, 1): "64x64 streamed",
    (13, 1, 34, 54, 47, 99, 3, 1, 1): "64x64 rounds, then streamed",
    (18, 1, 121, 51, 36, 37, 3, 1, 1): "64x128 streamed",
    (44, 1, 35, 46, 50, 45, 3, 1, 1): "64x128 rounds, then streamed",
    (37, 1, 151, 11, 41, 118, 3, 1, 1): "128x128 streamed",
    (45, 1, 172, 49, 30, 99, 1, 1, 0): "128x128 rounds, then streamed",
    (1, 1, 3, 40, 40, 64, 33, 1, 2): "64x64 ranges",  # 64-bit gathers
    (4, 1, 64, 26, 26, 32, 3, 1, 1): "32x128 ranges",
    (2, 2, 64, 9, 9, 72, 3, 1, 1): "64x64 whole",     # groups
    (2, 1, 3, 33, 31, 20, 3, 1, 1): "64x64 whole",    # 27 k
}
DATA_GRADIENTS = {
    (1, 1, 96, 13, 13, 1024, 1, 1, 0): "64x64 ranges",
    (45, 1, 99, 49, 30, 172, 1, 1, 0): "128x128 rounds, then streamed",
    (2, 1, 40, 7, 7, 300, 1, 1, 0): "64x64 ranges",
}


def _buffers(case, seed):
    batch, groups, cin, H, W, F, ks, s, p = case
    r = rng(seed)
    n = ref.conv_out_dim(H, ks, s, p) * ref.conv_out_dim(W, ks, s, p)
    x = r.integers(-4, 5, batch * cin * H * W).astype(np.float32)
    w = r.integers(-4, 5, F * (cin // groups) * ks * ks).astype(np.float32)
    d = r.integers(-4, 5, batch * F * n).astype(np.float32)
    return up(x), up(w), up(d)


def _forward(case, x, w, out):
    gpu.convolutionForward(*case, w, x, out)


def _data_gradient(case, d, w, out):
    gpu.convolutionDataGradient(*case, w, d, out)


def _plans():
    return [(c, _forward) for c in FORWARDS] + [(c, _data_gradient) for c in DATA_GRADIENTS]


def _kind(case, op):
    batch, groups, cin, H, W, F, ks, s, p = case
    n = batch * ref.conv_out_dim(H, ks, s, p) * ref.conv_out_dim(W, ks, s, p)
    m, k = (F, cin * ks * ks) if op is _forward else (cin, F)
    return tiling(m // groups, n, k // groups, groups, OWN, wide=ks > 32).kind


def _setup(case, op, seed=1):
    x, w, d = _buffers(case, seed)
    src, other = (x, d) if op is _forward else (d, x)
    return src, w, other, gpu.alloc(other.len)


def _stream(hip):
    s = C.c_void_p()
    hip.L.hipStreamCreateWithFlags.argtypes = [C.POINTER(C.c_void_p), C.c_uint]
    assert hip.L.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # hipStreamNonBlocking
    return s


@pytest.mark.parametrize("case,op", _plans(), ids=lambda v: v.__name__ if callable(v) else str(v))
def test_same_on_every_stream_and_in_a_graph(quiet, case, op):  # noqa: F811
    assert _kind(case, op) == (FORWARDS if op is _forward else DATA_GRADIENTS)[case]
    hip = Hip()
    src, w, other, out = _setup(case, op)
    like = np.empty(out.len, np.float32)
    op(case, src, w, out)
    want = down(out, like)
    s, graph, exe = _stream(hip), C.c_void_p(), C.c_void_p()
    try:
        gpu.fill(out, out.len, 0.0)
        gpu.sync()
        quiet.dkz_set_stream(s)
        op(case, src, w, out)
        np.testing.assert_array_equal(down(out, like), want)
        assert hip.hipStreamBeginCapture(s, 0) == 0
        gpu.fill(out, out.len, 0.0)
        op(case, src, w, out)
        assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0
        quiet.dkz_set_stream(None)
        assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, 0) == 0
        for _ in range(3):
            gpu.fill(out, out.len, 7.0)  # eager work between the replays
            gpu.sync()
            assert hip.hipGraphLaunch(exe, s) == 0
            assert hip.hipStreamSynchronize(s) == 0
            np.testing.assert_array_equal(down(out, like), want)
    finally:
        quiet.dkz_set_stream(None)
        gpu.sync()
        if exe.value:
            hip.hipGraphExecDestroy(exe)
        if graph.value:
            hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(s)
    for b in (src, w, other, out):
        gpu.free(b)


def test_overlapping_streams(quiet):  # noqa: F811
    """Three streams (the null one among them), each with its own layer and
    buffers, fed in turn without waiting: twenty accumulated passes each."""
    hip = Hip()
    plans = [((1, 1, 64, 52, 52, 128, 3, 1, 1), _forward), ((39, 1, 263, 13, 13, 153, 3, 1, 1), _forward),
             ((45, 1, 99, 49, 30, 172, 1, 1, 0), _data_gradient)]
    state = [_setup(c, op, 3 + i) for i, (c, op) in enumerate(plans)]
    want = []
    for (case, op), (src, w, _, out) in zip(plans, state):
        op(case, src, w, out)
        one = down(out, np.empty(out.len, np.float32))
        want.append(20 * one if op is _forward else one)  # the 1x1 data gradient overwrites
        gpu.fill(out, out.len, 0.0)
    gpu.sync()
    streams = [None, _stream(hip), _stream(hip)]
    try:
        for _ in range(20):
            for (case, op), (src, w, _, out), s in zip(plans, state, streams):
                quiet.dkz_set_stream(s)
                op(case, src, w, out)
        quiet.dkz_set_stream(None)
        gpu.sync()
        for (_, _, _, out), ref_out in zip(state, want):
            np.testing.assert_array_equal(down(out, np.empty(out.len, np.float32)), ref_out)
    finally:
        quiet.dkz_set_stream(None)
        gpu.sync()
        for s in streams[1:]:
            hip.hipStreamDestroy(s)
    for bufs in state:
        for b in bufs:
            gpu.free(b)


def test_two_threads_on_the_null_stream(quiet):  # noqa: F811
    """Two host threads, each with its own layer: a product and its reduction
    stay together."""
    import threading
    plans = [((1, 1, 64, 52, 52, 128, 3, 1, 1), _forward), ((1, 1, 512, 13, 13, 96, 3, 1, 1), _forward)]
    state = [_setup(c, op, 7 + i) for i, (c, op) in enumerate(plans)]
    errors = []

    def work(i):
        try:
            _lib.load().dkz_init(0)  # this thread's device
            (case, op), (src, w, _, out) = plans[i], state[i]
            for _ in range(200):
                op(case, src, w, out)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    want = []
    for (case, op), (src, w, _, out) in zip(plans, state):
        op(case, src, w, out)
        want.append(200 * down(out, np.empty(out.len, np.float32)))
        gpu.fill(out, out.len, 0.0)
    gpu.sync()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    gpu.sync()
    for (_, _, _, out), ref_out in zip(state, want):
        np.testing.assert_array_equal(down(out, np.empty(out.len, np.float32)), ref_out)
    for bufs in state:
        for b in bufs:
            gpu.free(b)
