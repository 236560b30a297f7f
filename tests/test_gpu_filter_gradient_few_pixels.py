"""fp32 filter gradients of fewer than 256 pixels: the kernel that shares the pixels out
among the eight waves of a work-group, some of which get none; a pixel, whole channel
tiles, ragged ones from 96 pixels on, strides, windows larger than the image, 1x1.

Bound: a sum of at most n products in fp32: (n + 4) 2^-24 of the sum of the products'
magnitudes (the sums of the waves are added on top: three steps).
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import DIRECTION, DTYPE
from test_gpu_parity import dev, oracle, oracle_params, uniform

pytestmark = pytest.mark.gpu

W = DIRECTION.FILTER_BACKPROP


@pytest.mark.parametrize("shape", [
    # batch, rows, cols, channels, features, window, stride, SAME
    (1, 1, 1, 64, 36, 3, 1, True),      # one pixel
    (1, 2, 1, 128, 64, 5, 1, True),
    (2, 7, 7, 64, 68, 7, 1, False),     # an image per pixel
    (3, 5, 5, 192, 20, 3, 2, True),
    (1, 5, 7, 64, 132, 1, 1, True),     # 35 pixels: shares that end inside
    (5, 3, 17, 128, 4, 3, 1, True),     # 255
    (1, 8, 12, 37, 53, 3, 1, True),     # 96 pixels, ragged: the first it takes
    (1, 5, 19, 37, 53, 3, 1, True),     # 95: the last of the other kernel
    (4, 6, 5, 99, 66, 5, 1, True),
    (3, 8, 10, 489, 320, 1, 1, True),
])
def test_few_pixels(shape):
    p = ops.conv_params(*shape)
    rng = np.random.default_rng(17 + shape[1])
    n_x, n_dy, _ = ops.conv_sizes(p, W)
    x, dy = uniform(rng, n_x), uniform(rng, n_dy)
    ref = oracle.conv2d_filter_backprop(x, dy, oracle_params(p, p.features),
                                        acc64=True).reshape(-1)
    norm = oracle.conv2d_filter_backprop(
        np.abs(x), np.abs(dy), oracle_params(p, p.features), acc64=True).reshape(-1)
    algorithm = ops.default_algorithm(p, W, DTYPE.F32)
    got = ops.conv2d(dev(x), dev(dy), p, W, algorithm)
    pixels = p.batch * p.out_rows * p.out_cols
    error = np.abs(got.cpu().numpy().reshape(-1).astype(np.float64) - ref)
    assert np.all(error <= (pixels + 4) * 2.0 ** -24 * norm)
    again = ops.conv2d(dev(x), dev(dy), p, W, algorithm)
    assert torch.equal(got.view(torch.int32), again.view(torch.int32))


@pytest.mark.parametrize("shape", [
    (1, 8, 12, 37, 53, 3, 1, True),
    (1, 5, 7, 64, 132, 3, 1, True),
    (5, 3, 17, 128, 4, 5, 1, True),
    (2, 9, 9, 36, 52, 3, 2, True),
    (8, 7, 7, 5, 100, 7, 2, True),      # few channels, many taps
    (8, 7, 7, 5, 98, 7, 2, True),
    (2, 14, 13, 64, 64, 3, 2, True),    # 98 pixels; and larger layers
    (4, 14, 14, 64, 128, 5, 2, True),
])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_borders_of_not_finite_gradients(shape, value):
    """A gradient in the corner belongs to the taps that meet the image there, not to
    those that meet its padding."""
    p = ops.conv_params(*shape)
    rng = np.random.default_rng(23 + shape[1])
    n_x, n_dy, _ = ops.conv_sizes(p, W)
    x, dy = uniform(rng, n_x), uniform(rng, n_dy)
    dy[1] = value
    dy[-2] = value
    ref = oracle.conv2d_filter_backprop(x, dy, oracle_params(p, p.features),
                                        acc64=True).reshape(-1)
    algorithm = ops.default_algorithm(p, W, DTYPE.F32)
    got = ops.conv2d(dev(x), dev(dy), p, W, algorithm).cpu().numpy().reshape(-1)
    finite = np.isfinite(ref)
    assert finite.any() and not finite.all()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    pixels = p.batch * p.out_rows * p.out_cols
    assert np.all(np.abs(got[finite] - ref[finite]) <=
                  2 * pixels * 2.0 ** -24 * np.sqrt(pixels))
