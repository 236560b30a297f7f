"""fp32 forward convolutions and input gradients at the sizes where the
gathering kernel can go wrong: edges of its tiles, ragged channel and feature
counts, stride classes with few, unequal or no taps, merged classes of a few
channels, reductions shared by work-groups, filters that are not 16-byte
aligned, bias and activation, infinite operands, launches recorded into a graph.

Bound: n products added in fp32, each addition rounding by at most 2^-24 of a
partial sum, which for the U[-1,1] operands here stays below twice the largest
output S: |gpu - ref| <= 2 n 2^-24 S.
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

# batch, rows, cols, channels, features, window, stride, same
SHAPES = [
    (2, 9, 7, 8, 8, 3, 1, True),        # the smallest pieces
    (1, 13, 11, 20, 30, 3, 2, True),    # features of no whole piece
    (3, 10, 13, 35, 45, 5, 1, False),   # odd counts: widened, 4-byte runs
    (2, 12, 15, 24, 40, 3, 3, True),    # nine classes
    (2, 15, 14, 40, 24, 2, 3, False),   # classes that no tap reaches
    (2, 16, 16, 64, 136, 1, 2, True),   # 1x1 strided: three empty classes
    (1, 16, 17, 32, 33, 1, 4, False),   # ... sixteen classes, odd features
    (1, 18, 18, 16, 16, 12, 1, True),   # the largest window
    (1, 20, 20, 8, 12, 13, 2, True),    # one larger: another kernel
    (1, 23, 23, 96, 129, 3, 1, True),   # one feature and one pixel past tiles
    (2, 7, 7, 480, 72, 3, 2, True),     # long reduction, few tiles: shared
    (9, 57, 43, 72, 96, 3, 2, True),    # many tiles, ragged rows
    (5, 31, 29, 84, 16, 1, 1, True),    # 1x1, reduction of no whole chunk
    (3, 40, 33, 100, 66, 1, 1, True),
    (40, 50, 51, 3, 32, 7, 2, True),    # merged classes, three channels
    (30, 47, 61, 3, 58, 3, 2, False),   # ... odd features, VALID
    (31, 50, 64, 1, 200, 5, 3, True),   # ... nine classes of one channel
    (20, 60, 60, 2, 40, 6, 4, True),    # ... sixteen of two
    (60, 45, 44, 4, 68, 2, 2, True),    # ... one tap per class
    (3, 21, 22, 35, 45, 1, 2, True),    # strided 1x1, odd: copied subsampled
    (2, 17, 19, 30, 66, 1, 3, False),   # ... even counts, VALID
    (20, 20, 21, 64, 203, 3, 1, True),  # many tiles, runs of odd features
    (9, 41, 43, 35, 133, 1, 2, True),   # large enough to be copied subsampled
    (3, 33, 35, 130, 66, 1, 3, False),
    (4, 40, 41, 32, 33, 1, 4, False),   # sixteen classes, odd features
    (13, 15, 19, 8, 135, 1, 2, True),   # short launches: the direct kernel
    (7, 45, 45, 6, 6, 1, 1, False),     # ... and its gradient
    (25, 14, 18, 56, 424, 1, 2, True),  # ... the implicit-GEMM kernel
    (1, 30, 30, 441, 52, 1, 1, True),   # ... its gradient
    (18, 18, 18, 36, 100, 3, 2, True),  # shared, or without a workspace whole
    (5, 37, 27, 32, 40, 3, 1, True),
]


def check(got, ref, n_products, what):
    got = np.asarray(got.cpu().numpy(), dtype=np.float64).reshape(-1)
    ref = np.asarray(ref, dtype=np.float64).reshape(-1)
    bound = 2 * n_products * 2.0**-24 * np.abs(ref).max()
    err = np.abs(got - ref)
    assert np.all(err <= bound), (what, err.max(), bound)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction", [DIRECTION.FORWARD,
                                       DIRECTION.INPUT_BACKPROP])
def test_conv_f32_shapes(shape, direction):
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    rng = np.random.default_rng(4300 + rows + channels + features)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a, b = uniform(rng, n_a), uniform(rng, n_b)
    ref = ORACLE_FN[direction](a, b, oracle_params(p, features), acc64=True)
    da, db = dev(a), dev(b)
    shifted = torch.empty(n_b + 1, device="cuda")[1:]
    shifted.copy_(db)
    n = window * window * (channels if direction == DIRECTION.FORWARD
                           else features)
    _, rec = ops.workspace_size(p, direction, ALGO.IM2COL)
    block = torch.full((rec + 4096,), 7.0, device="cuda")
    for fil, ws in ((db, None), (db, block[:rec] if rec else None),
                    (shifted, None)):
        guard = torch.full((n_out + 4096,), 7.0, device="cuda")
        got = ops.conv2d(da, fil, p, direction, ALGO.IM2COL, workspace=ws,
                         out=guard[:n_out])
        check(got, ref, n, (shape, direction, ws is None, fil is db))
        assert torch.all(guard[n_out:] == 7.0)
    assert torch.all(block[rec:] == 7.0)


@pytest.mark.parametrize("shape", [(3, 20, 21, 20, 30, 3, 2, True),
                                   (2, 7, 7, 480, 72, 3, 2, True),
                                   (5, 31, 29, 84, 16, 1, 1, True),
                                   (25, 14, 18, 56, 424, 1, 2, True),
                                   (13, 15, 19, 8, 135, 1, 2, True)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("relu", [False, True])
def test_conv_f32_bias_act(shape, relu):
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    rng = np.random.default_rng(4400 + rows)
    n_a, n_b, n_out = ops.conv_sizes(p, DIRECTION.FORWARD)
    a, b, bias = uniform(rng, n_a), uniform(rng, n_b), uniform(rng, features)
    ref = ORACLE_FN[DIRECTION.FORWARD](a, b, oracle_params(p, features),
                                       acc64=True)
    ref = ref.reshape(-1, features).astype(np.float64) + bias
    if relu:
        ref = np.maximum(ref, 0)
    got = ops.conv2d_bias_act(dev(a), dev(b), dev(bias), p, ALGO.IM2COL,
                              relu=relu)
    check(got, ref, window * window * channels + 1, (shape, relu))


# Merged classes (3x3, 7x7 and 5x5 windows, whole reductions and a shared one),
# classes of their own, forward windows over the border.
INFINITE = [
    ((30, 47, 61, 3, 58, 3, 2, True), DIRECTION.INPUT_BACKPROP),
    ((20, 50, 51, 3, 40, 7, 2, True), DIRECTION.INPUT_BACKPROP),
    ((20, 60, 60, 2, 40, 6, 4, True), DIRECTION.INPUT_BACKPROP),
    ((31, 50, 64, 1, 200, 5, 3, True), DIRECTION.INPUT_BACKPROP),
    ((1, 24, 24, 3, 512, 7, 2, True), DIRECTION.INPUT_BACKPROP),
    ((2, 12, 15, 24, 40, 3, 3, True), DIRECTION.INPUT_BACKPROP),
    ((2, 7, 7, 480, 72, 3, 2, True), DIRECTION.INPUT_BACKPROP),
    ((3, 10, 13, 35, 45, 5, 1, True), DIRECTION.FORWARD),
    ((2, 7, 7, 480, 70, 3, 2, True), DIRECTION.FORWARD),
    ((9, 57, 43, 72, 96, 3, 2, True), DIRECTION.FORWARD),
]


@pytest.mark.parametrize("shape,direction", INFINITE, ids=str)
@pytest.mark.parametrize("operand", [0, 1], ids=["tensor", "filter"])
def test_conv_f32_infinity_stays(shape, direction, operand):
    """An infinite value reaches the outputs that it is a factor of and no
    other: the finite rest is what it is without it."""
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    rng = np.random.default_rng(4700 + rows)
    n_a, n_b, _ = ops.conv_sizes(p, direction)
    a, b = uniform(rng, n_a), uniform(rng, n_b)
    if operand == 0:  # in the middle of an image
        forward = direction == DIRECTION.FORWARD
        r, c = (rows, cols) if forward else (p.out_rows, p.out_cols)
        a[(r // 2 * c + c // 2) * (channels if forward else features)] = np.inf
    else:             # the first tap, which the border pixels do not have
        b[0] = np.inf
    ref = ORACLE_FN[direction](a, b, oracle_params(p, features), acc64=True)
    ref = np.asarray(ref, dtype=np.float64).reshape(-1)
    got = ops.conv2d(dev(a), dev(b), p, direction, ALGO.IM2COL)
    ok = torch.from_numpy(np.isfinite(ref))
    assert ok.any() and not ok.all()
    assert torch.equal(torch.isfinite(got.cpu()), ok)
    check(got.cpu()[ok], ref[ok.numpy()], window * window *
          max(channels, features), (shape, direction, operand))


def test_conv_f32_bias_act_infinity_stays():
    shape = batch, rows, cols, channels, features, window, stride, same = (
        3, 20, 21, 20, 30, 3, 2, True)
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    rng = np.random.default_rng(4800)
    n_a, n_b, _ = ops.conv_sizes(p, DIRECTION.FORWARD)
    a, b, bias = uniform(rng, n_a), uniform(rng, n_b), uniform(rng, features)
    b[-1] = np.inf
    ref = ORACLE_FN[DIRECTION.FORWARD](a, b, oracle_params(p, features),
                                       acc64=True)
    ref = np.asarray(ref, dtype=np.float64).reshape(-1, features) + bias
    ref = np.maximum(ref, 0).reshape(-1)
    got = ops.conv2d_bias_act(dev(a), dev(b), dev(bias), p, ALGO.IM2COL,
                              relu=True)
    ok = torch.from_numpy(np.isfinite(ref))
    assert torch.equal(torch.isfinite(got.cpu()), ok) and not ok.all()
    check(got.cpu()[ok], ref[ok.numpy()], window * window * channels + 1, shape)


@pytest.mark.parametrize("shape,direction", [
    ((2, 7, 7, 480, 72, 3, 2, True), DIRECTION.FORWARD),
    ((2, 7, 7, 480, 72, 3, 2, True), DIRECTION.INPUT_BACKPROP),
    ((30, 47, 61, 3, 56, 3, 2, True), DIRECTION.INPUT_BACKPROP)],
    ids=str)
def test_conv_f32_captured(shape, direction):
    """Without a workspace a recorded launch takes no temporary."""
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    rng = np.random.default_rng(4500 + rows)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a, b = dev(uniform(rng, n_a)), dev(uniform(rng, n_b))
    out = torch.empty(n_out, device="cuda")
    ops.conv2d(a, b, p, direction, ALGO.IM2COL, out=out)
    n = window * window * (channels if direction == DIRECTION.FORWARD
                           else features)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        ops.conv2d(a, b, p, direction, ALGO.IM2COL, out=out)
    for seed in (1, 2, 3):
        a.copy_(dev(uniform(np.random.default_rng(seed), n_a)))
        want = ops.conv2d(a, b, p, direction, ALGO.IM2COL).double().cpu()
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        check(out, want.numpy(), n, (shape, direction, seed))
