"""Filter gradients whose channel or feature counts are rounded up in a copy:
either count or both odd, only one of them, first layers, every window, with the
queried workspace, without one, recorded into a graph, and with operands off
16-byte alignment.

Bound: n products added in fp32, each addition rounding by at most 2^-24 of a
partial sum, which for the U[-1,1] operands here stays below twice the largest
output S; binary16 rounds the result once more: |gpu - ref| <= 2 n 2^-24 S
(+ 2^-11 |ref| + 2^-24).
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_conv_f16_shapes import check_recorded
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

# batch, rows, cols, channels, features, window, stride, same
SHAPES = [
    (16, 28, 28, 65, 66, 3, 1, True),    # both
    (16, 28, 27, 64, 67, 3, 1, False),   # features only
    (16, 27, 28, 66, 64, 3, 1, True),    # channels only
    (5, 31, 30, 9, 35, 5, 1, True),      # the fewest channels that are rounded
    (20, 40, 41, 70, 33, 3, 2, True),
    (4, 112, 110, 3, 37, 7, 2, True),    # first layers, odd features
    (6, 90, 91, 4, 61, 5, 2, False),
    (6, 64, 64, 5, 42, 3, 1, True),
    (20, 100, 99, 3, 44, 3, 2, True),    # a multiple of 4, not of 8
    (10, 50, 50, 8, 33, 3, 1, True),     # the most channels that stay
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [DTYPE.F32, DTYPE.F16],
                         ids=["f32", "f16"])
def test_filter_gradient_widened(shape, dtype):
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    half = dtype == DTYPE.F16
    kind = torch.float16 if half else torch.float32
    rng = np.random.default_rng(4600 + rows + channels + features)
    n_x, n_dy, n_dw = ops.conv_sizes(p, DIRECTION.FILTER_BACKPROP)
    numpy_kind = np.float16 if half else np.float32
    x = uniform(rng, n_x).astype(numpy_kind)
    dy = uniform(rng, n_dy).astype(numpy_kind)
    ref = ORACLE_FN[DIRECTION.FILTER_BACKPROP](
        x.astype(np.float32), dy.astype(np.float32),
        oracle_params(p, features), acc64=True)
    ref = np.asarray(ref, dtype=np.float64).reshape(-1)
    n = batch * p.out_rows * p.out_cols
    bound = 2 * n * 2.0**-24 * np.abs(ref).max()
    if half:
        bound = bound + 2.0**-11 * np.abs(ref) + 2.0**-24
    dx, ddy = dev(x, kind), dev(dy, kind)
    shifted = torch.empty(n_dy + 1, dtype=kind, device="cuda")[1:]
    shifted.copy_(ddy)
    _, rec = ops.workspace_size(p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                                dtype)
    block = torch.full((rec + 4096,), 7.0, dtype=kind, device="cuda")
    for grad, ws in ((ddy, None), (ddy, block[:rec] if rec else None),
                     (shifted, None)):
        guard = torch.full((n_dw + 4096,), 7.0, dtype=kind, device="cuda")
        got = ops.conv2d(dx, grad, p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                         workspace=ws, out=guard[:n_dw])
        err = np.abs(got.double().cpu().numpy().reshape(-1) - ref)
        assert np.all(err <= bound), (shape, ws is None, err.max())
        assert torch.all(guard[n_dw:] == 7.0)
    assert torch.all(block[rec:] == 7.0)


@pytest.mark.parametrize("shape,dtype", [
    ((8, 112, 112, 3, 61, 7, 2, True), DTYPE.F32),
    ((20, 100, 99, 3, 42, 3, 2, True), DTYPE.F32),
    ((10, 50, 50, 8, 33, 3, 1, True), DTYPE.F32),
    ((16, 28, 28, 65, 66, 3, 1, True), DTYPE.F16),
    ((20, 100, 99, 3, 44, 3, 2, True), DTYPE.F16)], ids=str)
def test_filter_gradient_widened_recorded(shape, dtype):
    """The queried workspace holds all that the launches need."""
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    kind = torch.float16 if dtype == DTYPE.F16 else torch.float32
    n_x, n_dy, n_dw = ops.conv_sizes(p, DIRECTION.FILTER_BACKPROP)
    x = torch.empty(n_x, dtype=kind, device="cuda")
    dy = torch.empty(n_dy, dtype=kind, device="cuda")
    _, rec = ops.workspace_size(p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                                dtype)
    ws = torch.empty(rec, dtype=kind, device="cuda")

    def refill(seed):
        rng = np.random.default_rng(seed)
        x.copy_(dev(uniform(rng, n_x), kind))
        dy.copy_(dev(uniform(rng, n_dy), kind))

    refill(0)
    check_recorded(
        lambda out: ops.conv2d(x, dy, p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                               workspace=ws, out=out),
        refill, batch * p.out_rows * p.out_cols, (shape, dtype))
