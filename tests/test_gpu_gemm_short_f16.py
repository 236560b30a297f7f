"""Binary16 1x1 layers of few tiles, whose reduction the waves of a work-group
share: rows and columns that fill no tile, reductions shorter than all waves'
shares, not a multiple of them, and of more than one block of 1024.

Bound: one rounding to binary16 and n fp32 additions.
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION
from test_gpu_conv_f16_shapes import assert_rounded_once, check_recorded
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

# pixels, reduced, produced
SHAPES = [(1, 8, 8), (31, 24, 56), (33, 64, 64), (65, 128, 72), (40, 136, 200),
          (100, 264, 64), (70, 520, 136), (33, 1000, 40), (32, 1024, 64),
          (50, 1032, 128), (37, 2048, 72), (500, 16, 1000)]


def operands(pixels, reduced, produced, direction, seed):
    grad = direction == DIRECTION.INPUT_BACKPROP
    channels, features = (produced, reduced) if grad else (reduced, produced)
    p = ops.conv_params(1, 1, pixels, channels, features, 1, 1, True)
    rng = np.random.default_rng(seed + pixels + reduced)
    n_a, n_b, _ = ops.conv_sizes(p, direction)
    return p, (uniform(rng, n_a).astype(np.float16),
               uniform(rng, n_b).astype(np.float16))


def reference(p, direction, a, b):
    return np.asarray(ORACLE_FN[direction](
        a.astype(np.float32), b.astype(np.float32),
        oracle_params(p, p.features), acc64=True), dtype=np.float64).reshape(-1)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction",
                         [DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP])
def test_short_product(shape, direction):
    p, (a, b) = operands(*shape, direction, 7100)
    ref = reference(p, direction, a, b)
    guard = torch.full((ref.size + 4096,), 7.0, dtype=torch.float16,
                       device="cuda")
    got = ops.conv2d(dev(a, torch.float16), dev(b, torch.float16), p, direction,
                     ALGO.MATMUL, out=guard[:ref.size])
    assert_rounded_once(got.float().cpu().numpy(), ref, shape[1],
                        (shape, direction))
    assert torch.all(guard[ref.size:] == 7.0)


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[4], SHAPES[9]],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction",
                         [DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP])
def test_short_product_infinity_stays(shape, direction):
    p, (a, b) = operands(*shape, direction, 7200)
    a[-1], b[0] = np.inf, -np.inf  # the last pixel, one filter element
    ref = reference(p, direction, a, b)
    got = ops.conv2d(dev(a, torch.float16), dev(b, torch.float16), p, direction,
                     ALGO.MATMUL).float().cpu().numpy().reshape(-1)
    ok = np.isfinite(ref)
    assert ok.any() and not ok.all()
    assert np.array_equal(np.isfinite(got), ok)
    assert_rounded_once(got[ok], ref[ok], shape[1], (shape, direction))


@pytest.mark.parametrize("direction",
                         [DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP])
def test_short_product_recorded(direction):
    p, (a, b) = operands(100, 264, 64, direction, 7300)
    da, db = dev(a, torch.float16), dev(b, torch.float16)

    def refill(seed):
        rng = np.random.default_rng(seed)
        da.copy_(dev(uniform(rng, a.size), torch.float16).reshape(da.shape))
        db.copy_(dev(uniform(rng, b.size), torch.float16).reshape(db.shape))

    check_recorded(
        lambda out: ops.conv2d(da, db, p, direction, ALGO.MATMUL, out=out),
        refill, 264, direction)
