"""Binary16 forward convolutions and input gradients at the sizes where the
gathering kernel can go wrong: edges of its tiles, ragged channel and feature
counts, stride classes with few, unequal or no taps, reductions shared by
work-groups, filters that are not 16-byte aligned, infinite weights, launches
recorded into a graph; and short launches, which other kernels take.

Bound: the result is rounded to binary16 once (2^-11 of its magnitude) and its
n products are added in fp32, each addition rounding by at most 2^-24 of a
partial sum, which for the U[-1,1] operands here is of the size of the outputs:
|gpu - ref| <= 2^-11 |ref| + n 2^-24 S + 2^-24 (subnormals), S the largest |ref|.
"""
import ctypes

import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu


def assert_rounded_once(got, ref, n_products, what):
    got = np.asarray(got, dtype=np.float64).reshape(-1)
    ref = np.asarray(ref, dtype=np.float64).reshape(-1)
    size = np.abs(ref)
    bound = 2.0**-11 * size + n_products * 2.0**-24 * size.max() + 2.0**-24
    err = np.abs(got - ref)
    assert np.all(err <= bound), (what, err.max(), np.argmax(err - bound))


# batch, rows, cols, channels, features, window, stride, same
SHAPES = [
    (2, 9, 7, 8, 8, 1, 1, True),        # the smallest pieces
    (1, 13, 11, 20, 30, 3, 2, True),    # no multiples of 8; nothing full
    (3, 10, 13, 35, 45, 5, 1, False),   # odd counts: widened, 2-byte runs
    (2, 17, 16, 36, 68, 3, 1, True),    # multiples of 4: 8-byte runs
    (2, 12, 15, 24, 40, 3, 3, True),    # nine classes
    (2, 15, 14, 40, 24, 2, 3, False),   # classes that no tap reaches
    (2, 16, 16, 64, 136, 1, 2, True),   # 1x1 strided: three empty classes
    (1, 16, 17, 32, 33, 1, 4, False),   # ... sixteen classes, odd features
    (1, 18, 18, 16, 16, 12, 1, True),   # the largest window
    (1, 20, 20, 8, 12, 13, 2, True),    # one larger: another kernel
    (2, 20, 21, 64, 64, 13, 1, True),   # ... the LDS-tile kernel
    (2, 40, 41, 32, 64, 13, 2, True),   # ... fp32 copies
    (4, 16, 16, 96, 128, 3, 1, True),   # whole tiles of 128
    (1, 23, 23, 96, 129, 3, 1, True),   # one feature and one pixel past them
    (2, 7, 7, 512, 72, 3, 1, True),     # long reduction, few tiles: shared
    (5, 9, 9, 264, 264, 3, 2, True),    # ... by classes of unequal length
    (9, 57, 43, 72, 96, 3, 2, True),    # many tiles, ragged rows
    (16, 40, 40, 64, 200, 3, 2, True),  # tiles of 128 pixels and of 64
    (3, 21, 22, 35, 45, 1, 2, True),    # strided 1x1, odd: copied subsampled
    (2, 17, 19, 30, 66, 1, 3, False),   # ... even counts, VALID
    (20, 20, 21, 64, 203, 3, 1, True),  # many tiles, runs of odd features
    (5, 41, 43, 70, 65, 1, 2, True),    # large enough to be copied subsampled
    (3, 33, 35, 130, 66, 1, 3, False),
    (6, 40, 41, 64, 37, 1, 4, False),   # sixteen classes, odd features
    (4, 29, 29, 36, 44, 1, 1, True),    # short: the general kernel, no launch
    (3, 30, 28, 72, 20, 3, 2, True),    # ... in front of it; stride 2
    (1, 67, 50, 96, 3, 3, 3, True),     # ... the direct kernel's gradient
    (10, 58, 43, 6, 40, 1, 2, True),    # ... and forward
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction", [DIRECTION.FORWARD,
                                       DIRECTION.INPUT_BACKPROP])
def test_conv_f16_shapes(shape, direction):
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    rng = np.random.default_rng(4100 + rows + channels + features)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    ref = ORACLE_FN[direction](a.astype(np.float32), b.astype(np.float32),
                               oracle_params(p, features), acc64=True)
    da, db = dev(a, torch.float16), dev(b, torch.float16)
    shifted = torch.empty(n_b + 1, dtype=torch.float16, device="cuda")[1:]
    shifted.copy_(db)
    n = window * window * (channels if direction == DIRECTION.FORWARD
                           else features)
    _, rec = ops.workspace_size(p, direction, ALGO.IM2COL, DTYPE.F16)
    block = torch.full((rec + 4096,), 7.0, dtype=torch.float16, device="cuda")
    for fil, ws, at in ((db, None, 0), (db, block[:rec] if rec else None, 0),
                        (shifted, None, 0), (db, None, 1)):
        guard = torch.full((n_out + 4096,), 7.0, dtype=torch.float16,
                           device="cuda")
        got = ops.conv2d(da, fil, p, direction, ALGO.IM2COL, workspace=ws,
                         out=guard[at:at + n_out])
        assert_rounded_once(got.float().cpu().numpy(), ref, n,
                            (shape, direction, ws is None, fil is db, at))
        assert torch.all(guard[:at] == 7.0)
        assert torch.all(guard[at + n_out:] == 7.0)
    assert torch.all(block[rec:] == 7.0)


# The tiles of 256 pixels: packed filters (forward) and filters in place
# (gradients whose features fill whole pieces), whole chunks per tap or not,
# outputs in whole pieces or through LDS, a last tile with a remainder.
TILES = [
    ((33, 45, 23, 8, 16, 3, 1, True), 0, (256, 64)),
    ((17, 45, 23, 32, 130, 2, 1, True), 0, (256, 64)),
    ((33, 45, 23, 32, 16, 2, 1, True), 0, (256, 64)),
    ((17, 45, 23, 20, 130, 2, 1, True), 0, (256, 64)),
    ((33, 45, 23, 8, 65, 2, 1, True), 0, (256, 128)),
    ((33, 45, 23, 32, 65, 2, 1, True), 0, (256, 128)),
    ((9, 64, 40, 32, 136, 2, 1, True), 0, (256, 128)),
    ((9, 64, 40, 20, 136, 2, 1, True), 0, (256, 128)),
    ((66, 21, 23, 8, 32, 2, 3, True), 1, (256, 64)),
    ((66, 21, 23, 20, 16, 2, 3, True), 1, (256, 64)),
    ((66, 21, 23, 20, 65, 2, 3, True), 1, (256, 64)),
    ((66, 21, 23, 96, 32, 2, 3, True), 1, (256, 128)),
    ((66, 21, 23, 67, 32, 2, 3, True), 1, (256, 128)),
    ((66, 21, 23, 67, 16, 2, 3, True), 1, (256, 128)),
    ((66, 45, 23, 96, 65, 2, 3, True), 1, (256, 128)),
]


@pytest.mark.parametrize("shape,direction,tile", TILES, ids=str)
def test_conv_f16_large_tiles(shape, direction, tile):
    p = ops.conv_params(*shape)
    assert ops.gather_tile(p, direction, DTYPE.F16)[:2] == tile
    test_conv_f16_shapes(shape, direction)


def graph_node_types(graph):
    """The node types of a torch.cuda.CUDAGraph made with keep_graph=True."""
    hip = ctypes.CDLL("libamdhip64.so")
    raw = ctypes.c_void_p(graph.raw_cuda_graph())
    count = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * count.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(count)) == 0
    types = []
    for node in nodes:
        kind = ctypes.c_int()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node),
                                       ctypes.byref(kind)) == 0
        types.append(kind.value)
    return types


def check_recorded(call, refill, n_products, what):
    """Records call(out), which may launch kernels only, and compares three
    replays on refilled operands with eager calls."""
    out = call(None)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call(out)
    assert set(graph_node_types(graph)) == {0}, what  # hipGraphNodeTypeKernel
    graph.instantiate()
    for seed in (1, 2, 3):
        refill(seed)
        want = call(None).float().cpu().numpy()
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        # (both sides round once, and add in orders of their own)
        got = out.float().cpu().numpy()
        bound = 2 * (2.0**-11 * np.abs(want) + 2.0**-24 +
                     n_products * 2.0**-24 * np.abs(want).max())
        assert np.all(np.abs(got - want) <= bound), (what, seed)


@pytest.mark.parametrize("shape,direction", [
    ((2, 16, 16, 20, 32, 3, 1, True), DIRECTION.FORWARD),
    ((2, 16, 16, 20, 32, 3, 1, True), DIRECTION.INPUT_BACKPROP),
    ((9, 57, 43, 72, 96, 3, 2, True), DIRECTION.FORWARD),
    ((9, 57, 43, 72, 96, 3, 2, True), DIRECTION.INPUT_BACKPROP),
    ((2, 7, 7, 480, 72, 3, 2, True), DIRECTION.FORWARD),
    ((2, 7, 7, 480, 72, 3, 2, True), DIRECTION.INPUT_BACKPROP),
    ((2, 17, 16, 36, 68, 3, 1, True), DIRECTION.INPUT_BACKPROP),
    ((2, 12, 12, 33, 40, 3, 1, True), DIRECTION.FORWARD),
    ((2, 12, 12, 40, 33, 3, 1, True), DIRECTION.INPUT_BACKPROP)], ids=str)
def test_conv_f16_recorded_without_a_workspace(shape, direction):
    """Counts in multiples of 4, and small launches of any: kernels only."""
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a = torch.empty(n_a, dtype=torch.float16, device="cuda")
    b = torch.empty(n_b, dtype=torch.float16, device="cuda")

    def refill(seed):
        rng = np.random.default_rng(seed)
        a.copy_(dev(uniform(rng, n_a), torch.float16))
        b.copy_(dev(uniform(rng, n_b), torch.float16))

    refill(0)
    check_recorded(
        lambda out: ops.conv2d(a, b, p, direction, ALGO.IM2COL, out=out),
        refill, window * window * max(channels, features), (shape, direction))


@pytest.mark.parametrize("shape,direction", [
    ((9, 57, 43, 72, 96, 3, 2, True), DIRECTION.FORWARD),
    ((9, 57, 43, 72, 96, 3, 2, True), DIRECTION.INPUT_BACKPROP),
    ((2, 7, 7, 512, 72, 3, 1, True), DIRECTION.FORWARD),
    ((20, 20, 21, 64, 203, 3, 1, True), DIRECTION.FORWARD),
    ((20, 20, 21, 64, 203, 3, 1, True), DIRECTION.INPUT_BACKPROP),
    ((16, 80, 80, 128, 128, 3, 2, True), DIRECTION.FORWARD)], ids=str)
def test_conv_f16_infinite_filter_stays(shape, direction):
    """An infinite weight reaches the outputs that it is a factor of, and not
    those whose window has that tap outside the image."""
    batch, rows, cols, channels, features, window, stride, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, stride,
                        same)
    rng = np.random.default_rng(4150 + rows)
    n_a, n_b, _ = ops.conv_sizes(p, direction)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    b[0] = np.inf   # (the first tap ...
    b[-1] = np.inf  # ... and the last: stride 2 has padding on one side only)
    ref = ORACLE_FN[direction](a.astype(np.float32), b.astype(np.float32),
                               oracle_params(p, features), acc64=True)
    ref = np.asarray(ref, dtype=np.float64).reshape(-1)
    got = ops.conv2d(dev(a, torch.float16), dev(b, torch.float16), p, direction,
                     ALGO.IM2COL).float().cpu().numpy().reshape(-1)
    ok = np.isfinite(ref)
    assert ok.any() and not ok.all()
    assert np.array_equal(np.isfinite(got), ok)
    assert_rounded_once(got[ok], ref[ok], window * window *
                        max(channels, features), (shape, direction))


@pytest.mark.parametrize("m,k,n", [(32, 64, 64), (33, 40, 24), (257, 100, 130),
                                   (640, 1000, 30), (2588, 14, 56),
                                   (97, 1189, 338)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_matmul_f16_ragged(m, k, n, trans_b):
    rng = np.random.default_rng(4200 + m + k + n)
    a = uniform(rng, m * k).astype(np.float16)
    b = uniform(rng, k * n).astype(np.float16)
    bm = b.reshape(n, k).T if trans_b else b.reshape(k, n)
    ref = a.reshape(m, k).astype(np.float64) @ bm.astype(np.float64)
    got = ops.matmul(dev(a, torch.float16), dev(b, torch.float16), 1, m, k, n,
                     trans_b=trans_b)
    assert_rounded_once(got.float().cpu().numpy(), ref, k, (m, k, n, trans_b))


@pytest.mark.parametrize("m,k,n", [(257, 100, 130), (96, 1189, 40)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_matmul_f16_recorded(m, k, n, trans_b):
    """A reduction of no whole chunks of 64: kernels only."""
    a = torch.empty(m * k, dtype=torch.float16, device="cuda")
    b = torch.empty(k * n, dtype=torch.float16, device="cuda")

    def refill(seed):
        rng = np.random.default_rng(seed)
        a.copy_(dev(uniform(rng, m * k), torch.float16))
        b.copy_(dev(uniform(rng, k * n), torch.float16))

    refill(0)
    check_recorded(
        lambda out: ops.matmul(a, b, 1, m, k, n, trans_b=trans_b, out=out),
        refill, k, (m, k, n, trans_b))
