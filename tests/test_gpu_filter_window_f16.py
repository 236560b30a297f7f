"""Binary16 filter gradients of 3x3 and 5x5 windows on the kernel that keeps bands
of pixels in LDS, at the sizes where it can go wrong: bands of several rows and of
parts of a row, several images per band group, channel and feature counts that fill
no tile of 64, planes of a stride of 2, every padding.

Layers of fewer than 256 output pixels and at least 2^24 multiply-adds always take
it; the last ones take it by the estimate of its time.

Bound: one rounding to binary16 and n fp32 additions.
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_conv_f16_shapes import assert_rounded_once
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

# batch, rows, cols, channels, features, window, stride, same
SHAPES = [
    (1, 15, 17, 88, 120, 3, 1, True),     # ragged tiles
    (1, 1, 255, 64, 128, 3, 1, True),     # segments of one row
    (28, 3, 3, 72, 136, 3, 1, True),      # several images per group
    (1, 17, 17, 72, 128, 3, 1, False),    # no padding
    (1, 5, 160, 64, 128, 3, 2, True),     # planes in segments
    (4, 14, 16, 72, 120, 3, 2, True),     # padding on one side
    (4, 13, 15, 72, 136, 3, 2, True),     # ... on both
    (3, 18, 18, 96, 104, 3, 2, False),
    (1, 1, 250, 40, 72, 5, 1, True),
    (1, 15, 16, 56, 56, 5, 1, True),
    (2, 14, 14, 64, 56, 5, 1, False),
    (250, 1, 1, 64, 64, 5, 1, True),      # images smaller than the window
    (3, 111, 69, 144, 72, 3, 1, True),    # many bands, partial tiles summed
    (6, 42, 95, 216, 232, 3, 2, True),    # ... in planes
    (8, 74, 40, 64, 72, 5, 1, True),
    (1, 42, 55, 136, 200, 5, 1, True),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_filter_window_f16(shape):
    p = ops.conv_params(*shape)
    assert ops.lds_form_f16(p, DIRECTION.FILTER_BACKPROP) is not None
    rng = np.random.default_rng(6100 + shape[1] + shape[3])
    n_a, n_b, n_out = ops.conv_sizes(p, DIRECTION.FILTER_BACKPROP)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    ref = ORACLE_FN[DIRECTION.FILTER_BACKPROP](
        a.astype(np.float32), b.astype(np.float32),
        oracle_params(p, p.features), acc64=True)
    da, db = dev(a, torch.float16), dev(b, torch.float16)
    _, rec = ops.workspace_size(p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                                DTYPE.F16)
    assert rec > 0
    block = torch.full((rec + 4096,), 7.0, dtype=torch.float16, device="cuda")
    # (the last one: a filter off 8-byte alignment has other kernels)
    for ws, off in ((block[:rec], 0), (None, 0), (None, 1)):
        guard = torch.full((n_out + 4096,), 7.0, dtype=torch.float16,
                           device="cuda")
        got = ops.conv2d(da, db, p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                         workspace=ws, out=guard[off:off + n_out])
        assert_rounded_once(got.float().cpu().numpy(), ref,
                            p.batch * p.out_rows * p.out_cols, (shape, off))
        assert torch.all(guard[off + n_out:] == 7.0)
        assert torch.all(guard[:off] == 7.0)
    assert torch.all(block[rec:] == 7.0)


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[1], SHAPES[4], SHAPES[6],
                                   SHAPES[9]],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("operand", [0, 1])
def test_filter_window_f16_infinity_stays(shape, operand):
    """An infinite pixel reaches the elements of dW whose products hold it, and
    not those whose tap leaves the image there."""
    p = ops.conv_params(*shape)
    rng = np.random.default_rng(6200 + shape[1])
    n_a, n_b, _ = ops.conv_sizes(p, DIRECTION.FILTER_BACKPROP)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    # the image's first pixel, and one at its right border
    (a, b)[operand][0] = np.inf
    cols, each = ((p.in_cols, p.channels), (p.out_cols, p.features))[operand]
    (a, b)[operand][(cols - 1) * each + 5] = -np.inf
    ref = np.asarray(ORACLE_FN[DIRECTION.FILTER_BACKPROP](
        a.astype(np.float32), b.astype(np.float32),
        oracle_params(p, p.features), acc64=True), dtype=np.float64).reshape(-1)
    got = ops.conv2d(dev(a, torch.float16), dev(b, torch.float16), p,
                     DIRECTION.FILTER_BACKPROP,
                     ALGO.IM2COL).float().cpu().numpy().reshape(-1)
    ok = np.isfinite(ref)
    assert ok.any() and not ok.all()
    assert np.array_equal(np.isfinite(got), ok)
    assert_rounded_once(got[ok], ref[ok], p.batch * p.out_rows * p.out_cols,
                        (shape, operand))


@pytest.mark.parametrize("shape", [(4, 224, 224, 64, 64, 3, 1, True),
                                   (28, 101, 112, 88, 72, 3, 2, True),
                                   (8, 74, 40, 64, 72, 5, 1, True)],
                         ids=lambda s: "x".join(map(str, s)))
def test_filter_window_f16_infinities_of_many_splits(shape):
    """What an overflow of a scaled loss leaves: infinities among gradients, whose
    products with the zeros of a ReLU are NaNs by right, and beside the border, whose
    products with the padding are none.  Such a launch takes at most a few times as
    long as a finite one (30 for those of the border, in every image)."""
    p = ops.conv_params(*shape)
    assert ops.lds_form_f16(p, DIRECTION.FILTER_BACKPROP) > 4
    rng = np.random.default_rng(6300 + shape[1])
    n_a, n_b, _ = ops.conv_sizes(p, DIRECTION.FILTER_BACKPROP)
    a = np.maximum(uniform(rng, n_a), 0).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    _, rec = ops.workspace_size(p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                                DTYPE.F16)
    ws = torch.empty(rec, dtype=torch.float16, device="cuda")
    da, db = dev(a, torch.float16), dev(b, torch.float16)

    def run():
        return ops.conv2d(da, db, p, DIRECTION.FILTER_BACKPROP, ALGO.IM2COL,
                          workspace=ws)

    def least_ms():
        times = []
        for _ in range(6):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in "ab")
            start.record()
            run()
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times[1:])

    finite_ms = max(least_ms(), 0.03)
    images = b.reshape(p.batch, p.out_rows, p.out_cols, p.features)
    x = a.reshape(p.batch, p.in_rows, p.in_cols, p.channels)
    images[1, 5, 7, 3] = np.inf        # inside
    images[2, 0, p.out_cols - 1, 9] = -np.inf  # at the border
    x[0, 0, 0, 5] = np.inf
    x[p.batch - 1, p.in_rows - 1, 4, 60] = np.nan
    da, db = dev(a, torch.float16), dev(b, torch.float16)
    ref = np.asarray(ORACLE_FN[DIRECTION.FILTER_BACKPROP](
        a.astype(np.float32), b.astype(np.float32),
        oracle_params(p, p.features), acc64=True), dtype=np.float64).reshape(-1)
    got = run().float().cpu().numpy().reshape(-1)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    assert ok.any() and np.isnan(ref).any() and np.isinf(ref).any()
    assert_rounded_once(got[ok], ref[ok], p.batch * p.out_rows * p.out_cols,
                        shape)
    assert least_ms() < 10 * finite_ms
    db[:] = np.inf
    assert least_ms() < 10 * finite_ms
    images[:, 0, 3, :] = np.inf
    db = dev(b, torch.float16)
    assert least_ms() < 30 * finite_ms
