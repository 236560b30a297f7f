"""Performance cases: what a user of this library has it do, layer by layer.

A case is one layer of a convolutional network, run the way an inference
program or a training loop runs it through portdnn_amd.ops: parameters,
algorithm and workspace are settled once when the network is set up, every
pass then makes the calls on the tensors at hand.

  op = "conv"       mode "infer": the layer with bias and ReLU, through the
                    fused call in fp32 and as the three calls convolution,
                    bias add and ReLU in binary16 (which has no fused call);
                    mode "train": forward, input gradient and filter gradient.
  op = "depthwise"  the same two modes, the forward without bias.
  op = "pool"       mode "infer": forward; "train": forward and gradient.

Convolutions go through the library's default algorithm for their direction
and element type.  The ranges: batches of 1 to 128; images of 7x7 to 224x224;
3 (first layer) or 16 to 1024 channels; windows 1, 3, 5 and 7; strides 1 and
2; SAME and VALID padding; fp32 and binary16.
"""
import math

import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE, POOL_OP

_TYPES = {"f32": torch.float32, "f16": torch.float16}
_DTYPES = {"f32": DTYPE.F32, "f16": DTYPE.F16}
_DIRECTIONS = (DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP,
               DIRECTION.FILTER_BACKPROP)


def _conv(name, mode, dtype, batch, size, channels, features, window, stride,
          same=True):
    return {"name": name, "op": "conv", "mode": mode, "dtype": dtype,
            "batch": batch, "rows": size, "cols": size, "channels": channels,
            "features": features, "window": window, "stride": stride,
            "same": same}


def _depthwise(name, mode, dtype, batch, size, channels, stride):
    return {"name": name, "op": "depthwise", "mode": mode, "dtype": dtype,
            "batch": batch, "rows": size, "cols": size, "channels": channels,
            "window": 3, "stride": stride, "same": True}


def _pool(name, mode, kind, dtype, batch, size, channels, window, stride,
          same=True):
    return {"name": name, "op": "pool", "mode": mode, "kind": kind,
            "dtype": dtype, "batch": batch, "rows": size, "cols": size,
            "channels": channels, "window": window, "stride": stride,
            "same": same}


def listed():
    return [
        # One image through a 3x3 layer: serving at the lowest latency.
        _conv("infer_f32_3x3_b1", "infer", "f32", 1, 56, 64, 64, 3, 1),
        # A small serving batch through a channel-reducing 1x1 layer.
        _conv("infer_f16_1x1_b8", "infer", "f16", 8, 14, 1024, 256, 1, 1),
        # Training steps at the batch sizes of bench.py: the 3x3 layer ...
        _conv("train_f32_3x3_b32", "train", "f32", 32, 28, 128, 128, 3, 1),
        _conv("train_f16_3x3_b128", "train", "f16", 128, 14, 256, 256, 3, 1),
        # ... the expanding 1x1 layer, whose tensors are its cost ...
        _conv("train_f16_1x1_b128", "train", "f16", 128, 56, 64, 256, 1, 1),
        # ... the 3x3 layer that halves the image ...
        _conv("train_f16_3x3s2_b128", "train", "f16", 128, 56, 128, 128, 3, 2),
        # ... and the network's first layer, 7x7 on three channels.
        _conv("train_f16_stem_b128", "train", "f16", 128, 224, 3, 64, 7, 2),
        # A 5x5 layer with an odd batch, an odd image and channels that are
        # no power of two.
        _conv("train_f32_5x5_b17", "train", "f32", 17, 27, 96, 256, 5, 1),
        # Full-resolution images: the largest tensors.
        _conv("train_f16_3x3_224", "train", "f16", 16, 224, 64, 64, 3, 1),
        # Depthwise layers: an early large one, a late small one.
        _depthwise("train_f32_dw_b32", "train", "f32", 32, 112, 32, 1),
        _depthwise("train_f16_dw_b128", "train", "f16", 128, 14, 512, 1),
        # The pooling layer behind the first convolution.
        _pool("train_f32_maxpool_b32", "train", "max", "f32", 32, 112, 64, 3,
              2),
    ]


def _log(rng, low, high):
    """An integer between low and high, spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _channels(rng, low, high):
    """Mostly multiples of 16, as networks have them; some that are only
    multiples of 4, and a few of no kind."""
    c = _log(rng, low, high)
    step = rng.choice((16, 16, 16, 16, 16, 4, 4, 1))
    return max(low, c // step * step)


def _any(rng):
    dtype = rng.choice(("f32", "f16"))
    mode = rng.choice(("train", "train", "infer"))
    batch = _log(rng, 1, 128)
    family = rng.choice(("3x3", "3x3", "1x1", "1x1", "strided", "5x5", "stem",
                         "depthwise", "depthwise", "pool"))
    size = _log(rng, 7, 224)
    same = rng.random() < 0.8
    if family == "stem":
        case = _conv(None, mode, dtype, batch, _log(rng, 96, 224), 3,
                     _channels(rng, 32, 96), rng.choice((3, 7)), 2, same)
    elif family == "depthwise":
        case = _depthwise(None, mode, dtype, batch, size,
                          _channels(rng, 16, 1024), rng.choice((1, 1, 2)))
    elif family == "pool":
        window, stride = rng.choice(((3, 2), (3, 2), (2, 2), (3, 1)))
        case = _pool(None, mode, rng.choice(("max", "avg")), dtype, batch,
                     size, _channels(rng, 16, 1024), window, stride, same)
    else:
        window, stride = {"3x3": (3, 1), "1x1": (1, 1), "5x5": (5, 1),
                          "strided": (rng.choice((1, 3)), 2)}[family]
        case = _conv(None, mode, dtype, batch, size, _channels(rng, 16, 1024),
                     _channels(rng, 16, 1024), window, stride, same)
    case["cols"] = max(7, int(round(case["rows"] *
                                    rng.choice((1, 1, 1, 0.75, 1.3)))))
    del case["name"]
    return case


def _seconds(case):
    """What a pass costs at least, at round rates, to compare cases by."""
    w = work(case)
    rate = 1.2e14 if case["dtype"] == "f32" else 1.2e15
    return w["bytes"] / 5e12 + w["flops"] / rate


def draw(rng):
    most = max(_seconds(c) for c in listed())
    while True:
        case = _any(rng)
        if _seconds(case) <= most:
            return case


def _params(case):
    window, stride, same = case["window"], case["stride"], case["same"]
    if case["op"] == "conv":
        p = ops.ConvParams(channels=case["channels"],
                           features=case["features"])
    elif case["op"] == "depthwise":
        p = ops.DepthwiseParams(channels=case["channels"],
                                channel_multiplier=1)
    else:
        p = ops.PoolParams(channels=case["channels"])
    p.batch, p.in_rows, p.in_cols = case["batch"], case["rows"], case["cols"]
    p.window_rows = p.window_cols = window
    p.stride_rows = p.stride_cols = stride
    return ops.add_padding_to(p, same)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _TYPES[case["dtype"]]
    p = _params(case)
    x_shape = (p.batch, p.in_rows, p.in_cols, p.channels)
    features = case.get("features", p.channels)
    y_shape = (p.batch, p.out_rows, p.out_cols, features)

    def normal(shape, scale):
        return (torch.randn(shape, generator=g, device="cuda") *
                scale).to(dtype)

    s = {"case": case, "p": p}
    # Activations as a ReLU leaves them (an image is not), filters at the
    # scale that keeps activations at 1, gradients of a scaled loss.
    s["x"] = normal(x_shape, 1.0)
    if p.channels != 3:
        s["x"].relu_()
    s["y"] = torch.empty(y_shape, dtype=dtype, device="cuda")
    if case["op"] != "pool":
        taps = case["window"] ** 2
        fan_in = taps * (p.channels if case["op"] == "conv" else 1)
        w_shape = ((case["window"], case["window"], p.channels) +
                   ((features,) if case["op"] == "conv" else (1,)))
        s["w"] = normal(w_shape, math.sqrt(2.0 / fan_in))
    if case["mode"] == "train":
        s["dy"] = normal(y_shape, 0.1)
        s["dx"] = torch.empty(x_shape, dtype=dtype, device="cuda")
        if case["op"] != "pool":
            s["dw"] = torch.empty(w_shape, dtype=dtype, device="cuda")
    if case["op"] == "conv":
        if case["mode"] == "infer":
            s["bias"] = normal((features,), 0.1)
        directions = _DIRECTIONS if case["mode"] == "train" else \
            _DIRECTIONS[:1]
        dt = _DTYPES[case["dtype"]]
        s["algo"] = [ops.default_algorithm(p, d, dt) for d in directions]
        need = max(ops.workspace_size(p, d, a, dt)[1]
                   for d, a in zip(directions, s["algo"]))
        s["workspace"] = (torch.empty(need, dtype=dtype, device="cuda")
                          if need else None)
    if case["op"] == "pool":
        s["kind"] = POOL_OP.MAX if case["kind"] == "max" else POOL_OP.AVERAGE
    return s


def run(s):
    op, mode, p = s["case"]["op"], s["case"]["mode"], s["p"]
    x, y = s["x"], s["y"]
    if op == "conv":
        algo, ws = s["algo"], s["workspace"]
        if mode == "infer":
            if x.dtype == torch.float32:
                ops.conv2d_bias_act(x, s["w"], s["bias"], p, algo[0],
                                    relu=True, workspace=ws, out=y)
            else:
                ops.conv2d(x, s["w"], p, DIRECTION.FORWARD, algo[0],
                           workspace=ws, out=y)
                ops.binaryop(y, s["bias"], y.shape, s["bias"].shape,
                             ops.BINARY_OP.ADD, out=y)
                ops.pointwise_forward(y, ops.POINTWISE_OP.RELU, out=y)
            return {"y": y}
        ops.conv2d(x, s["w"], p, DIRECTION.FORWARD, algo[0], workspace=ws,
                   out=y)
        ops.conv2d(s["dy"], s["w"], p, DIRECTION.INPUT_BACKPROP, algo[1],
                   workspace=ws, out=s["dx"])
        ops.conv2d(x, s["dy"], p, DIRECTION.FILTER_BACKPROP, algo[2],
                   workspace=ws, out=s["dw"])
        return {"y": y, "dx": s["dx"], "dw": s["dw"]}
    if op == "depthwise":
        ops.depthwise_conv2d(x, s["w"], p, DIRECTION.FORWARD, out=y)
        if mode == "infer":
            return {"y": y}
        ops.depthwise_conv2d(s["dy"], s["w"], p, DIRECTION.INPUT_BACKPROP,
                             out=s["dx"])
        ops.depthwise_conv2d(x, s["dy"], p, DIRECTION.FILTER_BACKPROP,
                             out=s["dw"])
        return {"y": y, "dx": s["dx"], "dw": s["dw"]}
    ops.pooling_forward(x, p, s["kind"], out=y)
    if mode == "infer":
        return {"y": y}
    if s["kind"] == POOL_OP.MAX:
        ops.pooling_max_grad(x, y, s["dy"], p, s["kind"], dx=s["dx"])
    else:
        ops.pooling_avg_grad(s["dy"], p, dx=s["dx"])
    return {"y": y, "dx": s["dx"]}


def work(case):
    """Every tensor of every call read or written once; the multiply-adds of
    the convolutions (of a pooling: one operation per window element)."""
    p = _params(case)
    each = 4 if case["dtype"] == "f32" else 2
    x = p.batch * p.in_rows * p.in_cols * p.channels
    features = case.get("features", p.channels)
    y = p.batch * p.out_rows * p.out_cols * features
    taps = case["window"] ** 2
    train = case["mode"] == "train"
    if case["op"] == "pool":
        values = x + y
        if train:
            values += (2 * x + 2 * y) if case["kind"] == "max" else (x + y)
        return {"bytes": each * values, "flops": y * taps * (2 if train else 1)}
    w = taps * p.channels * (features if case["op"] == "conv" else 1)
    flops = 2 * y * taps * (p.channels if case["op"] == "conv" else 1)
    n = 3 if train else 1
    return {"bytes": each * n * (x + y + w), "flops": n * flops}


def tolerance(case):
    # About four times the largest errors seen against the same layers in 64
    # bits, over the listed cases and sixty drawn ones: fp32 9.8e-7 in the
    # 2-norm and 7.3e-6 in one value, binary16 3.1e-4 and 1.0e-3 (one rounding
    # of the result, and of the two steps behind it for bias and ReLU).
    if case["dtype"] == "f32":
        return {"rel": 4e-6, "max": 3e-5}
    return {"rel": 1.2e-3, "max": 4e-3}
