"""Binary16 convolutions of one to four channels at stride 2 at the sizes where
the kernels for them can go wrong: every half-size tap count (windows 2 to 8 with
their paddings), features that fill no block, rows of an odd number of values,
bands and pixel blocks with remainders, several images per work-group.

Bound: as for the other binary16 convolutions, one rounding to binary16 and n
fp32 additions.
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_conv_f16_shapes import assert_rounded_once
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

DIRECTIONS = [DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP,
              DIRECTION.FILTER_BACKPROP]

# batch, rows, cols, channels, features, window, same
SHAPES = [
    (2, 34, 40, 3, 64, 7, True),     # four half-size taps
    (1, 39, 37, 3, 64, 7, False),    # odd rows and columns, no padding
    (3, 33, 71, 3, 40, 5, True),     # three; features past a block of 32
    (2, 64, 66, 3, 32, 3, True),     # two
    (1, 35, 131, 3, 96, 3, False),   # pixel blocks and chunks with remainders
    (2, 31, 30, 3, 96, 7, True),     # the most features
    (2, 30, 47, 1, 8, 7, True),      # one channel, one eighth of a block
    (1, 21, 22, 2, 24, 6, False),    # an even window
    (2, 25, 23, 4, 48, 4, True),
    (1, 26, 28, 4, 16, 8, True),     # five half-size taps: other kernels
    (2, 27, 29, 2, 72, 2, True),
    (1, 224, 224, 3, 64, 7, True),
    (70, 19, 18, 3, 64, 7, True),
    (600, 7, 9, 3, 32, 3, True),     # more images than work-groups
]


def make(shape, seed):
    batch, rows, cols, channels, features, window, same = shape
    p = ops.conv_params(batch, rows, cols, channels, features, window, 2, same)
    return p, np.random.default_rng(seed + rows + cols + features)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction", DIRECTIONS)
def test_few_channels_f16(shape, direction):
    p, rng = make(shape, 5100)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    ref = ORACLE_FN[direction](a.astype(np.float32), b.astype(np.float32),
                               oracle_params(p, p.features), acc64=True)
    window = p.window_rows * p.window_cols
    n = {DIRECTION.FORWARD: window * p.channels,
         DIRECTION.INPUT_BACKPROP: window * p.features,
         DIRECTION.FILTER_BACKPROP: p.batch * p.out_rows * p.out_cols}[direction]
    da, db = dev(a, torch.float16), dev(b, torch.float16)
    _, rec = ops.workspace_size(p, direction, ALGO.IM2COL, DTYPE.F16)
    block = torch.full((rec + 4096,), 7.0, dtype=torch.float16, device="cuda")
    for ws in (None, block[:rec] if rec else None):
        guard = torch.full((n_out + 4096,), 7.0, dtype=torch.float16,
                           device="cuda")
        got = ops.conv2d(da, db, p, direction, ALGO.IM2COL, workspace=ws,
                         out=guard[:n_out])
        assert_rounded_once(got.float().cpu().numpy(), ref, n,
                            (shape, direction, ws is None))
        assert torch.all(guard[n_out:] == 7.0)
    assert torch.all(block[rec:] == 7.0)


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[1], SHAPES[4], SHAPES[7]],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction", DIRECTIONS)
def test_few_channels_f16_infinity_stays(shape, direction):
    """An infinite pixel reaches the outputs whose window holds it and no other:
    the finite rest is what it is without the pixel."""
    p, rng = make(shape, 5200)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    # (the filter gradient: the last column that a window reaches, met by the
    # last pixel of a row only in its last column tap)
    if direction == DIRECTION.FILTER_BACKPROP:
        col = min(p.in_cols - 1,
                  2 * (p.out_cols - 1) + p.window_cols - 1 - p.pad_cols)
        row = 2 * (p.out_rows // 2)
        at = (row * p.in_cols + col) * p.channels
    else:
        cols = p.in_cols if direction == DIRECTION.FORWARD else p.out_cols
        rows = p.in_rows if direction == DIRECTION.FORWARD else p.out_rows
        each = p.channels if direction == DIRECTION.FORWARD else p.features
        at = ((rows // 2) * cols + cols // 2) * each
    a[at] = np.inf
    ref = ORACLE_FN[direction](a.astype(np.float32), b.astype(np.float32),
                               oracle_params(p, p.features), acc64=True)
    ref = np.asarray(ref).reshape(-1)
    got = ops.conv2d(dev(a, torch.float16), dev(b, torch.float16), p, direction,
                     ALGO.IM2COL).float().cpu().numpy().reshape(-1)
    assert np.isfinite(ref).any() and not np.isfinite(ref).all()
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    ok = np.isfinite(ref)
    assert_rounded_once(got[ok], ref[ok], max(
        p.window_rows * p.window_cols * max(p.channels, p.features),
        p.batch * p.out_rows * p.out_cols), (shape, direction))


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[2], SHAPES[3], SHAPES[6],
                                   SHAPES[12]],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction", DIRECTIONS[:2])
def test_few_channels_f16_infinite_filter_stays(shape, direction):
    """An infinite weight reaches the outputs that it is a factor of, and not
    those whose window has that tap outside the image."""
    p, rng = make(shape, 5300)
    n_a, n_b, _ = ops.conv_sizes(p, direction)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    b[0], b[-1] = np.inf, -np.inf  # the first tap and the last
    ref = ORACLE_FN[direction](a.astype(np.float32), b.astype(np.float32),
                               oracle_params(p, p.features), acc64=True)
    ref = np.asarray(ref).reshape(-1)
    got = ops.conv2d(dev(a, torch.float16), dev(b, torch.float16), p, direction,
                     ALGO.IM2COL).float().cpu().numpy().reshape(-1)
    ok = np.isfinite(ref)
    assert ok.any() and not ok.all()
    assert np.array_equal(np.isfinite(got), ok)
    assert_rounded_once(got[ok], ref[ok], p.window_rows * p.window_cols *
                        max(p.channels, p.features), (shape, direction))
