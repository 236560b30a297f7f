"""fp32 layers large enough for the gathering kernel's tiles with operands split
into bfloat16 parts: filters in place and packed, whole and broken chunks per tap,
ragged tiles, stride classes, shared reductions, bias and activation, infinities,
the largest and very small values.

Bound: n products added in fp32 as in the other fp32 convolutions; the products of
parts left out are below 2^-23 of a product, two roundings (2^-26 in the root mean
square).
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_conv_f32_shapes import check
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

F, I = DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP
# batch, rows, cols, channels, features, window, stride, same; direction; tile
CASES = [
    ((6, 99, 101, 112, 256, 3, 2, True), F, (128, 128)),  # whole chunks
    ((6, 99, 101, 112, 256, 3, 2, True), I, (128, 128)),  # ... four classes
    ((8, 70, 52, 16, 336, 5, 1, True), F, (128, 128)),    # one chunk per tap
    ((8, 70, 52, 16, 335, 5, 1, True), F, (128, 128)),    # packed, odd features
    ((14, 37, 35, 132, 100, 5, 1, False), F, (128, 128)), # broken chunks
    ((6, 41, 39, 132, 100, 5, 1, True), F, (128, 128)),   # ... shared reduction
    ((6, 41, 39, 101, 132, 5, 1, True), I, (128, 128)),   # ... odd columns
    ((6, 41, 39, 100, 133, 5, 1, True), I, (128, 128)),   # a copied source
    ((68, 26, 26, 71, 320, 3, 1, True), F, (128, 64)),    # ... the smaller tile
]
IDS = ["x".join(map(str, c[0])) + "fi"[c[1] == I] for c in CASES]


def operands(shape, direction, seed):
    p = ops.conv_params(*shape)
    rng = np.random.default_rng(seed + shape[1])
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    return p, uniform(rng, n_a), uniform(rng, n_b), n_out


def reference(p, direction, a, b):
    return np.asarray(ORACLE_FN[direction](
        a, b, oracle_params(p, p.features), acc64=True)).reshape(-1)


def products(p, direction):
    return p.window_rows * p.window_cols * (
        p.channels if direction == F else p.features)


@pytest.mark.parametrize("shape,direction,tile", CASES, ids=IDS)
def test_split_operands(shape, direction, tile):
    p, a, b, n_out = operands(shape, direction, 3300)
    assert ops.gather_tile(p, direction, DTYPE.F32)[:2] == tile
    ref = reference(p, direction, a, b)
    _, rec = ops.workspace_size(p, direction, ALGO.IM2COL, DTYPE.F32)
    block = torch.full((rec + 1024,), 7.0, device="cuda")
    da, db = dev(a), dev(b)
    for ws in (block[:rec], None):
        guard = torch.full((n_out + 1024,), 7.0, device="cuda")
        got = ops.conv2d(da, db, p, direction, ALGO.IM2COL, workspace=ws,
                         out=guard[:n_out])
        check(got, ref, products(p, direction), (shape, direction))
        assert torch.all(guard[n_out:] == 7.0)
    assert torch.all(block[rec:] == 7.0)
    # (closer to 64 bits than additions in fp32: 5e-7 and more at these lengths)
    error = got.cpu().numpy().astype(np.float64).reshape(-1) - ref
    assert np.linalg.norm(error) <= 4e-7 * np.linalg.norm(ref.astype(np.float64))


def test_split_operands_with_bias_and_relu():
    shape = CASES[0][0]
    p, a, b, _ = operands(shape, F, 3400)
    bias = uniform(np.random.default_rng(3), p.features)
    ref = reference(p, F, a, b).reshape(-1, p.features) + bias
    got = ops.conv2d_bias_act(dev(a), dev(b), dev(bias), p, ALGO.IM2COL,
                              relu=True)
    check(got, np.maximum(ref, 0), products(p, F) + 1, shape)


@pytest.mark.parametrize("shape,direction,tile", [CASES[0], CASES[1], CASES[5],
                                                  CASES[7]],
                         ids=[IDS[i] for i in (0, 1, 5, 7)])
@pytest.mark.parametrize("operand", [0, 1])
def test_split_operands_of_any_size(shape, direction, tile, operand):
    """Infinite and NaN values, the largest finite one, and ones whose parts the
    matrix units would take for zero."""
    p, a, b, n_out = operands(shape, direction, 3500)
    (a, b)[operand][:2] = np.inf, np.nan
    (a, b)[operand][-1] = np.finfo(np.float32).max
    # the last but one image (a filter has none): sums of 2^-110
    each = a.size // p.batch
    a[-2 * each:-each] *= np.float32(2.0**-112)
    ref = reference(p, direction, a, b)
    got = ops.conv2d(dev(a), dev(b), p, direction,
                     ALGO.IM2COL).cpu().numpy().reshape(-1)
    ok = np.isfinite(ref)
    assert ok.any() and not ok.all()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    n = products(p, direction)
    image = n_out // p.batch
    tiny = np.zeros(n_out, dtype=bool)
    tiny[-2 * image:-image] = True
    for part in (tiny & ok & (np.abs(ref) < 1e-30),
                 ~tiny & ok & (np.abs(ref) < 1e30)):
        assert part.any()
        error = np.abs(got[part].astype(np.float64) - ref[part])
        assert error.max() <= 2 * n * 2.0**-24 * np.abs(ref[part]).max()


@pytest.mark.parametrize("shape,direction,tile", [CASES[0], CASES[1], CASES[5],
                                                  CASES[8]],
                         ids=[IDS[i] for i in (0, 1, 5, 8)])
@pytest.mark.parametrize("small,large", [(-110, 10), (-115, 15), (-120, 20),
                                         (-130, 100), (-50, -60)])
@pytest.mark.parametrize("operand", [0, 1])
def test_split_operands_small_beside_large(shape, direction, tile, small, large,
                                           operand):
    """Operands whose later parts the matrix units would take for zero, with
    partners that make ordinary sums of them, and operands whose products come near
    the least: what the parts cannot hold is not missing from the sum.

    Bound: every addition rounds half a unit of a partial sum, which grows with the
    square root of its length."""
    p, a, b, _ = operands(shape, direction, 3600)
    both = []
    for k, v in enumerate((a, b)):
        v = np.where(v < 0, -1, 1) * (1 + np.abs(v) * np.float32(0.999))
        both.append(np.ldexp(v, small if k == operand else large)
                    .astype(np.float32))
    a, b = both
    ref = reference(p, direction, a, b).astype(np.float64)
    got = ops.conv2d(dev(a), dev(b), p, direction,
                     ALGO.IM2COL).cpu().numpy().reshape(-1).astype(np.float64)
    error = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert error <= np.sqrt(products(p, direction)) * 2.0**-24
