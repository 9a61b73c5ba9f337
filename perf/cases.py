"""Performance cases of the tensor-op layer: the layer passes a darknet program runs through `darknet_zig_amd.gpu`.

Each case is one pass of one layer (or of one direction of it) through the
public entry points, on tensors the program already holds on the GPU:

  conv_layer   a convolutional layer's forward: fill, convolution, batch norm and activation in place
  conv_fwd     a convolution's forward product alone (the layer's zero fill, then the product)
  conv_bwd     a convolution's backward: weight gradient and data gradient
  connected    a connected layer's forward and backward (its three gemms, bias and activation)
  bn_fwd       a batch-norm layer's training forward with its activation
  bn_bwd       a batch-norm layer's backward with its activation, as one call or as the ops the reference's layer issues
  head         a classifier's end: global average pool, softmax with cross-entropy, and back
  maxpool      a max-pool layer's forward and backward
  update       a layer's weight update: SGD with momentum and decay, or Adam, and its biases and scales
  residual     a shortcut layer's forward and backward

Tensors are fp32 NCHW, the framework's only element type. Gradients arrive
from the layer above: a pass that works on a gradient in place first takes it
into the layer's own buffer with `gpu.copy`, and gradients that accumulate
start from `gpu.fill`, as a network's step clears them.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from darknet_zig_amd import gpu
from darknet_zig_amd.activations import Activation

LEAKY, LINEAR, LOGISTIC = int(Activation.leaky), int(Activation.linear), int(Activation.logistic)
ACTS = {"leaky": LEAKY, "linear": LINEAR, "logistic": LOGISTIC}

# Caps on a drawn case: bytes and flops of a pass, below the largest listed ones.
MAX_BYTES = 1.6e9
MAX_FLOPS = 6.0e10


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # One image through a 3x3 layer of a detector: the smallest call of a serving loop, a few launches.
        dict(name="infer_1x64x52", kind="conv_layer", train=False, batch=1, c=64, hw=52, filters=128, ksize=3, stride=1),
        # The 3x3 layer of a 224-input classifier at a training batch: the ordinary convolution.
        dict(name="conv_fwd_64x128x56", kind="conv_fwd", batch=64, c=128, hw=56, filters=128, ksize=3, stride=1),
        # A detector's deepest 3x3 layer, 13x13 maps (169 positions: no multiple of four): the largest products.
        dict(name="conv_bwd_32x512x13", kind="conv_bwd", batch=32, c=512, hw=13, filters=1024, ksize=3, stride=1),
        # A connected layer before a classifier: products with short rows and a long inner dimension, TN/NT/NN.
        dict(name="connected_256x4096", kind="connected", batch=256, inputs=4096, outputs=1000),
        # Batch-norm forward with leaky at a small-image training batch: a few microseconds of memory traffic.
        dict(name="bn_fwd_128x32x32", kind="bn_fwd", act="leaky", batch=128, filters=32, hw=32),
        # The same pass on 13x13 maps, where a channel's rows start at any alignment.
        dict(name="bn_fwd_64x512x13", kind="bn_fwd", act="leaky", batch=64, filters=512, hw=13),
        # Batch-norm backward as the reference's layer issues it, op by op: the headline chain.
        dict(name="bn_bwd_64x128x56", kind="bn_bwd", act="leaky", fused=False, batch=64, filters=128, hw=56),
        # Batch-norm backward in one call on 13x13 maps.
        dict(name="bn_bwd_64x1024x13", kind="bn_bwd", act="leaky", fused=True, batch=64, filters=1024, hw=13),
        # The end of a 1000-class classifier: 7x7 maps to probabilities, loss and gradient.
        dict(name="head_256x1000x7", kind="head", batch=256, classes=1000, hw=7),
        # 2x2 max pooling of a large batch, both directions: the largest tensors.
        dict(name="maxpool_256x512x28", kind="maxpool", batch=256, c=512, hw=28, size=2, stride=2),
        # The SGD update of a 25M-weight layer.
        dict(name="sgd_25m", kind="update", adam=False, weights=25_000_000, filters=1024),
        # A residual block's shortcut where the map halves and the channels double.
        dict(name="residual_64x256x28", kind="residual", batch=64, c=256, hw=28, half=True),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["conv_layer", "conv_fwd", "conv_bwd", "connected", "bn_fwd", "bn_bwd", "head", "maxpool", "update",
                       "residual"])
    if kind in ("conv_layer", "conv_fwd", "conv_bwd"):
        k = rng.choice([1, 3, 3])
        case = dict(kind=kind, batch=_log(rng, 1, 64), c=_log(rng, 3, 1024), hw=_log(rng, 7, 208),
                    filters=_log(rng, 16, 1024), ksize=k, stride=rng.choice([1, 1, 1, 2]) if k == 3 else 1)
        if kind == "conv_layer":
            case["train"] = rng.random() < 0.4
        return case
    if kind == "connected":
        return dict(kind=kind, batch=_log(rng, 1, 256), inputs=_log(rng, 64, 4096), outputs=_log(rng, 10, 4096))
    if kind in ("bn_fwd", "bn_bwd"):
        case = dict(kind=kind, act=rng.choice(["leaky", "leaky", "linear"]), batch=_log(rng, 1, 128),
                    filters=_log(rng, 16, 1024), hw=_log(rng, 7, 112))
        if kind == "bn_bwd":
            case["fused"] = rng.random() < 0.6
        return case
    if kind == "head":
        return dict(kind=kind, batch=_log(rng, 1, 256), classes=_log(rng, 10, 2000), hw=_log(rng, 3, 14))
    if kind == "maxpool":
        size, stride = rng.choice([(2, 2), (2, 2), (3, 2), (2, 1), (5, 1), (9, 1), (13, 1)])
        return dict(kind=kind, batch=_log(rng, 1, 256), c=_log(rng, 16, 512), hw=_log(rng, 13, 26 if stride == 1 else 112),
                    size=size, stride=stride)
    if kind == "update":
        return dict(kind=kind, adam=rng.random() < 0.3, weights=_log(rng, 400, 25_000_000), filters=_log(rng, 16, 1024))
    return dict(kind=kind, batch=_log(rng, 1, 64), c=_log(rng, 16, 512), hw=2 * _log(rng, 4, 56), half=rng.random() < 0.4)


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= MAX_BYTES and w["flops"] <= MAX_FLOPS and w["bytes"] >= 4e4:
            return case


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------


def _conv(case):
    """(batch, channels, hw, filters, ksize, stride, pad, out_hw) of a convolution."""
    k, s, hw = case["ksize"], case["stride"], case["hw"]
    pad = k // 2
    return case["batch"], case["c"], hw, case["filters"], k, s, pad, (hw + 2 * pad - k) // s + 1


def _pool(case):
    """(hw, out_hw, pad) of a max pool; the layer's padding is size - 1."""
    pad = case["size"] - 1
    return case["hw"], (case["hw"] + pad - case["size"]) // case["stride"] + 1, pad


def work(case):
    kind = case["kind"]
    flops = 0.0
    if kind in ("conv_layer", "conv_fwd", "conv_bwd"):
        b, c, hw, f, k, s, _, oh = _conv(case)
        x, w, y = b * c * hw * hw, f * c * k * k, b * f * oh * oh
        one = 2.0 * f * c * k * k * b * oh * oh
        if kind == "conv_layer":  # input and weights in; output and the layer's x (and x_norm) out
            floats, flops = x + w + (3 if case["train"] else 2) * y, one
        elif kind == "conv_fwd":
            floats, flops = x + w + y, one
        else:  # delta, input and weights in; weight updates (read and written) and input delta out
            floats, flops = y + 2 * x + 3 * w, 2 * one
    elif kind == "connected":
        b, n, m = case["batch"], case["inputs"], case["outputs"]
        floats, flops = 2 * b * n + 3 * n * m + 3 * b * m, 6.0 * b * n * m
    elif kind == "bn_fwd":  # input; output, x, x_norm
        floats = 4 * case["batch"] * case["filters"] * case["hw"] ** 2
    elif kind == "bn_bwd":  # incoming delta, output, x, x_norm; delta
        floats = (5 if case["act"] != "linear" else 4) * case["batch"] * case["filters"] * case["hw"] ** 2
    elif kind == "head":  # maps in and their gradient out; truth in; pooled, probabilities, delta, loss, pooled delta out
        n = case["batch"] * case["classes"]
        floats = 2 * n * case["hw"] ** 2 + 6 * n
    elif kind == "maxpool":  # input; output, indexes; delta; the input's gradient
        hw, oh, _ = _pool(case)
        floats = case["batch"] * case["c"] * (2 * hw * hw + 3 * oh * oh)
    elif kind == "update":  # w and its gradient read and written, Adam's m and v too
        floats = (8 if case["adam"] else 4) * case["weights"] + 8 * case["filters"]
    else:  # residual: input and add in, output out; delta in, the layer's delta and both inputs' gradients out
        n, na = _residual(case)
        floats = 5 * n + 2 * na
    return {"bytes": 4.0 * floats, "flops": flops}


def _residual(case):
    """Elements of the block's output and of the earlier layer's output."""
    b, c, hw = case["batch"], case["c"], case["hw"]
    na = b * c * hw * hw
    return (b * 2 * c * (hw // 2) ** 2 if case["half"] else na), na


def tolerance(case):
    kind = case["kind"]
    if kind in ("maxpool", "update", "residual"):
        return "exact"  # elementwise, copies, first maxima, and sums in a fixed order
    # About four times the error against 64 bits that fp32 sums and roundings show over the ranges above.
    if kind.startswith("conv"):  # up to 1.2e-6 over sums of 9216 products
        return {"rel": 5e-6, "max": 2e-4}
    if kind == "connected":  # up to 5e-7 over sums of 4096 products
        return {"rel": 2e-6, "max": 8e-5}
    return {"rel": 5e-7, "max": 2e-5}  # sums in f64, a few roundings an element: 1e-7


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


class _Rand:
    """Seeded fp32 draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(std).add_(mean)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)


def _zeros(*shape):
    return torch.zeros(*shape, device="cuda")


def _leaky(x):
    return torch.where(x > 0, x, 0.1 * x)


def _inputs(case, seed):
    """The pass's input tensors, from the seed alone."""
    r, kind = _Rand(seed), case["kind"]
    t = {}
    if kind in ("conv_layer", "conv_fwd", "conv_bwd"):
        b, c, hw, f, k, s, _, oh = _conv(case)
        fan = c * k * k
        # The layer below ends in a leaky activation of normalised values.
        t["input"] = _leaky(r.normal(b, c, hw, hw))
        t["weights"] = r.normal(f, c, k, k, std=math.sqrt(2.0 / fan))
        if kind == "conv_bwd":
            t["delta"] = r.normal(b, f, oh, oh, std=0.05)
        if kind == "conv_layer":
            t["scales"], t["biases"] = r.uniform(f, lo=0.5, hi=1.5), r.normal(f, std=0.1)
            t["rolling_mean"], t["rolling_variance"] = r.normal(f, std=0.2), r.uniform(f, lo=0.5, hi=1.5)
    elif kind == "connected":
        b, n, m = case["batch"], case["inputs"], case["outputs"]
        t["input"] = _leaky(r.normal(b, n))
        t["weights"] = r.normal(m, n, std=math.sqrt(2.0 / n))
        t["biases"] = r.normal(m, std=0.1)
        t["incoming"] = r.normal(b, m, std=0.05)
    elif kind in ("bn_fwd", "bn_bwd"):
        b, f, hw = case["batch"], case["filters"], case["hw"]
        mu, sd = r.normal(1, f, 1, 1, std=0.3), r.uniform(1, f, 1, 1, lo=0.5, hi=1.5)
        t["x"] = r.normal(b, f, hw, hw).mul_(sd).add_(mu)
        t["scales"], t["biases"] = r.uniform(f, lo=0.5, hi=1.5), r.normal(f, std=0.1)
        t["rolling_mean"], t["rolling_variance"] = r.normal(f, std=0.2), r.uniform(f, lo=0.5, hi=1.5)
        if kind == "bn_bwd":  # what the forward pass left behind
            m, v = t["x"].mean((0, 2, 3)), t["x"].var((0, 2, 3))
            t["mean"], t["variance"] = m, v
            t["x_norm"] = (t["x"] - m.view(1, -1, 1, 1)).mul_(1.0 / (v.sqrt() + 1e-6).view(1, -1, 1, 1))
            y = t["x_norm"] * t["scales"].view(1, -1, 1, 1)
            y += t["biases"].view(1, -1, 1, 1)
            t["output"] = _leaky(y) if case["act"] == "leaky" else y
            t["incoming"] = r.normal(b, f, hw, hw)
    elif kind == "head":
        b, n, hw = case["batch"], case["classes"], case["hw"]
        t["input"] = r.normal(b, n, hw, hw, std=4.0)
        pick = torch.randint(0, n, (b,), generator=r.g, device="cuda")
        t["truth"] = F.one_hot(pick, n).float()
    elif kind == "maxpool":
        b, c = case["batch"], case["c"]
        hw, oh, _ = _pool(case)
        t["input"] = r.uniform(b, c, hw, hw, lo=-1.0, hi=1.0)
        t["delta"] = r.uniform(b, c, oh, oh, lo=-1.0, hi=1.0)
    elif kind == "update":
        n, f = case["weights"], case["filters"]
        t["w"], t["dw"] = r.normal(n, std=0.05), r.normal(n, std=0.05)
        for name in ("biases", "scales"):
            t[name], t[name + "_updates"] = r.normal(f, std=0.1), r.normal(f, std=0.05)
        if case["adam"]:
            t["m"], t["v"] = r.normal(n, std=0.01), r.uniform(n, lo=1e-5, hi=1e-3)
    else:
        b, c, hw = case["batch"], case["c"], case["hw"]
        shape = (b, 2 * c, hw // 2, hw // 2) if case["half"] else (b, c, hw, hw)
        t["input"], t["add"], t["incoming"] = r.normal(*shape), r.normal(b, c, hw, hw), r.normal(*shape)
    return t


def _buffers(case, t):
    """The layer's own buffers: outputs, gradients and statistics."""
    kind = case["kind"]
    o = {}
    if kind in ("conv_layer", "conv_fwd"):
        b, _, _, f, _, _, _, oh = _conv(case)
        o["output"] = _zeros(b, f, oh, oh)
        if kind == "conv_layer":
            o["x"] = _zeros(b, f, oh, oh)
            if case["train"]:
                o["x_norm"], o["mean"], o["variance"] = _zeros(b, f, oh, oh), _zeros(f), _zeros(f)
    elif kind == "conv_bwd":
        o["weight_updates"], o["input_delta"] = torch.zeros_like(t["weights"]), torch.zeros_like(t["input"])
    elif kind == "connected":
        for name in ("output", "delta"):
            o[name] = torch.zeros_like(t["incoming"])
        o["bias_updates"], o["weight_updates"] = torch.zeros_like(t["biases"]), torch.zeros_like(t["weights"])
        o["input_delta"] = torch.zeros_like(t["input"])
    elif kind == "bn_fwd":
        for name in ("out", "x_copy", "x_norm"):
            o[name] = torch.zeros_like(t["x"])
        o["mean"], o["variance"] = torch.zeros_like(t["scales"]), torch.zeros_like(t["scales"])
    elif kind == "bn_bwd":
        o["delta"] = torch.zeros_like(t["x"])
        for name in ("bias_updates", "scale_updates", "mean_delta", "variance_delta"):
            o[name] = torch.zeros_like(t["scales"])
    elif kind == "head":
        for name in ("pooled", "prob", "delta", "loss", "pooled_delta"):
            o[name] = torch.zeros_like(t["truth"])
        o["input_delta"] = torch.zeros_like(t["input"])
    elif kind == "maxpool":
        o["output"], o["input_delta"] = torch.zeros_like(t["delta"]), torch.zeros_like(t["input"])
        o["indexes"] = torch.zeros(t["delta"].shape, dtype=torch.int32, device="cuda")
    elif kind == "residual":
        o["output"], o["delta"], o["input_delta"] = (torch.zeros_like(t["input"]) for _ in range(3))
        o["add_delta"] = torch.zeros_like(t["add"])
    return o


def prepare(case, seed):
    if not gpu.active():
        gpu.init(0)
    tensors = _inputs(case, seed)
    tensors.update(_buffers(case, tensors))
    bufs = {name: gpu.Buf(t.data_ptr(), t.numel()) for name, t in tensors.items()}
    return {"case": case, "t": tensors, "b": bufs}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def _pick(t, *names):
    return {name: t[name] for name in names}


def _run_conv_layer(case, t, b):
    n, c, hw, f, k, s, pad, oh = _conv(case)
    gpu.fill(b["output"], n * f * oh * oh, 0.0)
    gpu.convolutionForward(n, 1, c, hw, hw, f, k, s, pad, b["weights"], b["input"], b["output"])
    train = case["train"]
    gpu.batchnormForward(n, f, oh * oh, LEAKY, train, b["output"], b["output"], b["x"], b.get("x_norm"), b.get("mean"),
                         b.get("variance"), b["rolling_mean"], b["rolling_variance"], b["scales"], b["biases"])
    names = ["output", "x"] + (["x_norm", "mean", "variance", "rolling_mean", "rolling_variance"] if train else [])
    return _pick(t, *names)


def _run_conv_fwd(case, t, b):
    n, c, hw, f, k, s, pad, oh = _conv(case)
    gpu.fill(b["output"], n * f * oh * oh, 0.0)
    gpu.convolutionForward(n, 1, c, hw, hw, f, k, s, pad, b["weights"], b["input"], b["output"])
    return _pick(t, "output")


def _run_conv_bwd(case, t, b):
    n, c, hw, f, k, s, pad, _ = _conv(case)
    gpu.convolutionWeightGradient(n, 1, c, hw, hw, f, k, s, pad, b["delta"], b["input"], b["weight_updates"])
    if k != 1:  # a 1x1 layer's gradient overwrites, the others add to the network's cleared one
        gpu.fill(b["input_delta"], n * c * hw * hw, 0.0)
    gpu.convolutionDataGradient(n, 1, c, hw, hw, f, k, s, pad, b["weights"], b["delta"], b["input_delta"])
    return _pick(t, "weight_updates", "input_delta")


def _run_connected(case, t, b):
    n, i, o = case["batch"], case["inputs"], case["outputs"]
    gpu.fill(b["output"], n * o, 0.0)
    gpu.gemm(False, True, n, o, i, 1.0, b["input"], i, b["weights"], i, 1.0, b["output"], o)
    gpu.addBias(b["output"], b["biases"], n, o, 1)
    gpu.activateArray(b["output"], n * o, LOGISTIC)
    gpu.copy(n * o, b["incoming"], b["delta"])
    gpu.gradientArray(b["output"], n * o, LOGISTIC, b["delta"])
    gpu.backwardBias(b["bias_updates"], b["delta"], n, o, 1)
    gpu.gemm(True, False, o, i, n, 1.0, b["delta"], o, b["input"], i, 1.0, b["weight_updates"], i)
    gpu.fill(b["input_delta"], n * i, 0.0)
    gpu.gemm(False, False, n, i, o, 1.0, b["delta"], o, b["weights"], i, 1.0, b["input_delta"], i)
    return _pick(t, "output", "delta", "bias_updates", "weight_updates", "input_delta")


def _run_bn_fwd(case, t, b):
    gpu.batchnormForward(case["batch"], case["filters"], case["hw"] ** 2, ACTS[case["act"]], True, b["x"], b["out"],
                         b["x_copy"], b["x_norm"], b["mean"], b["variance"], b["rolling_mean"], b["rolling_variance"],
                         b["scales"], b["biases"])
    return _pick(t, "out", "x_copy", "x_norm", "mean", "variance", "rolling_mean", "rolling_variance")


def _run_bn_bwd(case, t, b):
    n, f, s, act = case["batch"], case["filters"], case["hw"] ** 2, ACTS[case["act"]]
    gpu.copy(n * f * s, b["incoming"], b["delta"])
    if case["fused"]:
        gpu.batchnormBackward(n, f, s, act, b["output"], b["delta"], b["x"], b["x_norm"], b["mean"], b["variance"],
                              b["scales"], b["bias_updates"], b["scale_updates"], b["mean_delta"], b["variance_delta"])
    else:
        gpu.gradientArray(b["output"], n * f * s, act, b["delta"])
        gpu.backwardBias(b["bias_updates"], b["delta"], n, f, s)
        gpu.backwardScale(b["x_norm"], b["delta"], n, f, s, b["scale_updates"])
        gpu.scaleBias(b["delta"], b["scales"], n, f, s)
        gpu.meanDelta(b["delta"], b["variance"], n, f, s, b["mean_delta"])
        gpu.varianceDelta(b["x"], b["delta"], b["mean"], b["variance"], n, f, s, b["variance_delta"])
        gpu.normalizeDelta(b["x"], b["mean"], b["variance"], b["mean_delta"], b["variance_delta"], n, f, s, b["delta"])
    return _pick(t, "delta", "bias_updates", "scale_updates", "mean_delta", "variance_delta")


def _run_head(case, t, b):
    n, k, hw = case["batch"], case["classes"], case["hw"]
    gpu.forwardAvgpool(n * k, hw, hw, k, b["input"], b["pooled"])
    gpu.softmaxLayerForward(n, k, 1, 1.0, b["pooled"], b["truth"], b["prob"], b["delta"], b["loss"])
    gpu.fill(b["pooled_delta"], n * k, 0.0)
    gpu.axpy(n * k, 1.0, b["delta"], b["pooled_delta"])
    gpu.fill(b["input_delta"], n * k * hw * hw, 0.0)
    gpu.backwardAvgpool(n * k, hw, hw, k, b["input_delta"], b["pooled_delta"])
    return _pick(t, "pooled", "prob", "delta", "loss", "pooled_delta", "input_delta")


def _run_maxpool(case, t, b):
    n, c, size, stride = case["batch"], case["c"], case["size"], case["stride"]
    hw, oh, pad = _pool(case)
    gpu.forwardMaxpool(n * c * oh * oh, hw, hw, c, stride, size, pad, b["input"], b["output"], b["indexes"])
    gpu.fill(b["input_delta"], n * c * hw * hw, 0.0)
    gpu.backwardMaxpool(n * c * hw * hw, hw, hw, c, stride, size, pad, b["delta"], b["input_delta"], b["indexes"])
    return _pick(t, "output", "indexes", "input_delta")


# A training step of batch 64: learning rate 1e-3, momentum 0.9, weight decay 5e-4.
BATCH, RATE, MOMENTUM, DECAY = 64, 1e-3, 0.9, 5e-4
B1, B2, EPS, STEP = 0.9, 0.999, 1e-7, 10


def _run_update(case, t, b):
    n, f = case["weights"], case["filters"]
    for name in ("biases", "scales"):
        gpu.axpy(f, RATE / BATCH, b[name + "_updates"], b[name])
        gpu.scal(f, MOMENTUM, b[name + "_updates"])
    out = ["w", "dw", "biases", "scales", "biases_updates", "scales_updates"]
    if case["adam"]:
        gpu.adamUpdate(b["w"], b["dw"], b["m"], b["v"], B1, B2, EPS, DECAY, RATE, n, BATCH, STEP)
        out += ["m", "v"]
    else:
        gpu.axpy(n, -DECAY * BATCH, b["w"], b["dw"])
        gpu.axpy(n, RATE / BATCH, b["dw"], b["w"])
        gpu.scal(n, MOMENTUM, b["dw"])
    return _pick(t, *out)


def _run_residual(case, t, b):
    batch, c, hw = case["batch"], case["c"], case["hw"]
    c2, hw2 = (2 * c, hw // 2) if case["half"] else (c, hw)
    n, na = _residual(case)
    gpu.copy(n, b["input"], b["output"])
    gpu.shortcut(batch, hw, hw, c, b["add"], hw2, hw2, c2, 1.0, 1.0, b["output"])
    gpu.activateArray(b["output"], n, LEAKY)
    gpu.copy(n, b["incoming"], b["delta"])
    gpu.gradientArray(b["output"], n, LEAKY, b["delta"])
    gpu.fill(b["input_delta"], n, 0.0)
    gpu.axpy(n, 1.0, b["delta"], b["input_delta"])
    gpu.fill(b["add_delta"], na, 0.0)
    gpu.shortcut(batch, hw2, hw2, c2, b["delta"], hw, hw, c, 1.0, 1.0, b["add_delta"])
    return _pick(t, "output", "delta", "input_delta", "add_delta")


_RUN = {
    "conv_layer": _run_conv_layer, "conv_fwd": _run_conv_fwd, "conv_bwd": _run_conv_bwd, "connected": _run_connected,
    "bn_fwd": _run_bn_fwd, "bn_bwd": _run_bn_bwd, "head": _run_head, "maxpool": _run_maxpool, "update": _run_update,
    "residual": _run_residual,
}


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](case, state["t"], state["b"])


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------


def _f32(x):
    """A constant as the entry points take it (float)."""
    return float(torch.tensor(x, dtype=torch.float32))


def _act64(x, act):
    if act == "leaky":
        return torch.where(x > 0, x, _f32(0.1) * x)
    return torch.sigmoid(x) if act == "logistic" else x


def _chan(v):
    return v.view(1, -1, 1, 1)


def _conv64(t, case):
    """The convolution image by image (an im2col in f64 would not fit at once)."""
    n, _, _, f, k, s, pad, oh = _conv(case)
    w = t["weights"].double().reshape(f, -1)
    out = torch.empty(n, f, oh * oh, dtype=torch.float64, device="cuda")
    for i in range(n):
        col = F.unfold(t["input"][i:i + 1].double(), k, padding=pad, stride=s)[0]
        torch.mm(w, col, out=out[i])
    return out.view(n, f, oh, oh)


def _bn64(x, t, act, train):
    """(output, x_norm, mean, variance, rolling_mean, rolling_variance) of a batch-norm forward."""
    rm, rv = t["rolling_mean"].double(), t["rolling_variance"].double()
    m, v = (x.mean((0, 2, 3)), x.var((0, 2, 3), correction=1)) if train else (rm, rv)
    xn = (x - _chan(m)) / (_chan(v).sqrt() + 1e-6)
    y = _act64(xn * _chan(t["scales"].double()) + _chan(t["biases"].double()), act)
    keep, add = _f32(0.99), _f32(0.01)
    return y, xn, m, v, rm * keep + add * m, rv * keep + add * v


def _exact_conv_layer(case, t):
    x = _conv64(t, case)
    y, xn, m, v, rm, rv = _bn64(x, t, "leaky", case["train"])
    out = {"output": y, "x": x}
    if case["train"]:
        out.update(x_norm=xn, mean=m, variance=v, rolling_mean=rm, rolling_variance=rv)
    return out


def _exact_conv_fwd(case, t):
    return {"output": _conv64(t, case)}


def _exact_conv_bwd(case, t):
    n, c, hw, f, k, s, pad, oh = _conv(case)
    w = t["weights"].double().reshape(f, -1)
    dw = torch.zeros_like(w)
    dx = torch.empty(n, c, hw, hw, dtype=torch.float64, device="cuda")
    for i in range(n):
        d = t["delta"][i].double().reshape(f, -1)
        col = F.unfold(t["input"][i:i + 1].double(), k, padding=pad, stride=s)[0]
        dw += torch.mm(d, col.t().contiguous())
        dx[i] = F.fold(torch.mm(w.t().contiguous(), d)[None], (hw, hw), k, padding=pad, stride=s)[0]
    return {"weight_updates": dw.view(f, c, k, k), "input_delta": dx}


def _exact_connected(case, t):
    x, w = t["input"].double(), t["weights"].double()
    y = torch.sigmoid(torch.mm(x, w.t().contiguous()) + t["biases"].double())
    d = t["incoming"].double() * (1 - y) * y
    return {"output": y, "delta": d, "bias_updates": d.sum(0), "weight_updates": torch.mm(d.t().contiguous(), x),
            "input_delta": torch.mm(d, w)}


def _exact_bn_fwd(case, t):
    x = t["x"].double()
    y, xn, m, v, rm, rv = _bn64(x, t, case["act"], True)
    return {"out": y, "x_copy": x, "x_norm": xn, "mean": m, "variance": v, "rolling_mean": rm, "rolling_variance": rv}


def _exact_bn_bwd(case, t):
    x, d, v = t["x"].double(), t["incoming"].double(), t["variance"].double() + _f32(1e-5)
    if case["act"] == "leaky":
        d = torch.where(t["output"] > 0, d, _f32(0.1) * d)
    bias, scale = d.sum((0, 2, 3)), (d * t["x_norm"].double()).sum((0, 2, 3))
    d = d * _chan(t["scales"].double())
    xm = x - _chan(t["mean"].double())
    md = -d.sum((0, 2, 3)) / v.sqrt()
    vd = -0.5 * (d * xm).sum((0, 2, 3)) * v ** -1.5
    count = x.numel() // x.shape[1]
    delta = d / _chan(v.sqrt()) + (2.0 / count) * _chan(vd) * xm + _chan(md) / count
    return {"delta": delta, "bias_updates": bias, "scale_updates": scale, "mean_delta": md, "variance_delta": vd}


def _exact_head(case, t):
    p = t["input"].double().mean((2, 3))
    prob, truth = torch.softmax(p, 1), t["truth"].double()
    d = truth - prob
    back = (d / case["hw"] ** 2)[:, :, None, None].expand(t["input"].shape)
    loss = torch.where(truth != 0, -torch.log_softmax(p, 1), torch.zeros_like(p))
    return {"pooled": p, "prob": prob, "delta": d, "loss": loss, "pooled_delta": d, "input_delta": back.contiguous()}


def _exact_maxpool(case, t):
    size, stride = case["size"], case["stride"]
    hw, oh, pad = _pool(case)
    before, need = pad // 2, (oh - 1) * stride + size
    x = F.pad(t["input"].double(), (before, max(0, need - hw - before)) * 2, value=-math.inf)
    y, at = F.max_pool2d(x, size, stride, return_indices=True)
    wide = x.shape[3]
    y, at = y[:, :, :oh, :oh], at[:, :, :oh, :oh]
    flat = (at // wide - before) * hw + at % wide - before  # within the plane
    grad = torch.zeros(case["batch"] * case["c"], hw * hw, dtype=torch.float64, device="cuda")
    grad.scatter_add_(1, flat.reshape(grad.shape[0], -1), t["delta"].double().reshape(grad.shape[0], -1))
    plane = torch.arange(grad.shape[0], device="cuda").view(case["batch"], case["c"], 1, 1) * (hw * hw)
    return {"output": y.contiguous(), "indexes": (flat + plane).int(), "input_delta": grad.view(t["input"].shape)}


def _exact_update(case, t):
    t = {k: v.double() for k, v in t.items()}
    rate, keep = _f32(RATE / BATCH), _f32(MOMENTUM)
    out = {}
    for name in ("biases", "scales"):
        out[name] = t[name] + rate * t[name + "_updates"]
        out[name + "_updates"] = keep * t[name + "_updates"]
    d = t["dw"] + _f32(-DECAY * BATCH) * t["w"]
    if case["adam"]:
        b1, b2 = _f32(B1), _f32(B2)
        m, v = b1 * t["m"] + (1 - b1) * d, b2 * t["v"] + (1 - b2) * d * d
        step = _f32(RATE) * (m / (1 - b1 ** STEP)) / ((v / (1 - b2 ** STEP)).sqrt() + _f32(EPS))
        out.update(w=t["w"] + step, dw=torch.zeros_like(d), m=m, v=v)
    else:
        out.update(w=t["w"] + rate * d, dw=keep * d)
    return out


def _exact_residual(case, t):
    x, add, d = t["input"].double(), t["add"].double(), t["incoming"].double()
    c = case["c"]
    y = x.clone()
    y[:, :c] += add[:, :, ::2, ::2] if case["half"] else add
    d = torch.where(y > 0, d, _f32(0.1) * d)
    back = torch.zeros_like(add)
    if case["half"]:
        back[:, :, ::2, ::2] = d[:, :c]
    else:
        back += d
    return {"output": _act64(y, "leaky"), "delta": d, "input_delta": d, "add_delta": back}


_EXACT = {
    "conv_layer": _exact_conv_layer, "conv_fwd": _exact_conv_fwd, "conv_bwd": _exact_conv_bwd,
    "connected": _exact_connected, "bn_fwd": _exact_bn_fwd, "bn_bwd": _exact_bn_bwd, "head": _exact_head,
    "maxpool": _exact_maxpool, "update": _exact_update, "residual": _exact_residual,
}


def exact(case, seed):
    return _EXACT[case["kind"]](case, _inputs(case, seed))
