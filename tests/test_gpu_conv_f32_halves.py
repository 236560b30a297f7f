"""fp32 convolutions whose operands are taken apart into two binary16 values: every
tile, ragged pixels, channels and features, strips of columns, windows of 2 to 49
taps, strides, bias and activation, prepared filters; values that binary16's range
does not hold beside each other, infinities and NaNs.

Bound: n products added in fp32, as in the other fp32 convolutions.  Taken apart, an
operand is off by at most 2^-23 of itself and a product by 2^-22 of the two products
of low parts; both are roundings of single products of either sign, and add
2^-22 sqrt(n) of the sum's norm at the most.
"""
import ctypes

import numpy as np
import pytest
import torch

from portdnn_amd import capi, ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_conv_f32_shapes import check
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

F, I = DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP
TILED, WINO = ALGO.IM2COL, ALGO.WINOGRAD
# batch, rows, cols, channels, features, window, stride, same; direction; tag; tile
CASES = [
    ((8, 30, 29, 160, 132, 3, 1, True), F, TILED, (60, 128)),   # two image rows
    ((8, 30, 29, 160, 132, 3, 1, True), I, TILED, (60, 128)),   # ragged channels
    ((9, 41, 43, 100, 64, 3, 1, True), F, WINO, (64, 64)),
    ((40, 8, 8, 256, 132, 3, 1, True), I, TILED, (64, 64)),     # whole images
    ((3, 50, 60, 256, 160, 2, 1, True), F, TILED, (120, 64)),   # four taps
    ((3, 50, 60, 256, 160, 2, 1, True), I, TILED, (75, 128)),   # strips
    ((9, 41, 43, 100, 68, 4, 1, False), F, TILED, (60, 128)),   # sixteen taps
    ((1, 80, 104, 112, 224, 3, 1, True), F, WINO, (240, 32)),
    ((6, 57, 61, 40, 36, 7, 1, True), F, TILED, (93, 64)),      # 49 taps
    ((4, 27, 27, 96, 256, 5, 1, True), F, TILED, (56, 64)),     # 25 taps
    ((16, 27, 27, 96, 256, 5, 1, True), F, TILED, (126, 128)),
    ((40, 33, 31, 64, 64, 3, 1, True), F, WINO, (176, 64)),     # several tiles each
    ((12, 37, 39, 128, 256, 3, 2, True), F, TILED, (60, 128)),  # stride 2
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


def launch(p, direction, tag, a, b, **kw):
    _, rec = ops.workspace_size(p, direction, tag, DTYPE.F32)
    ws = torch.full((rec + 1024,), 7.0, device="cuda")
    out = ops.conv2d(dev(a), dev(b), p, direction, tag, workspace=ws[:rec], **kw)
    assert torch.all(ws[rec:] == 7.0)
    return out


@pytest.mark.parametrize("shape,direction,tag,tile", CASES, ids=IDS)
def test_taken_apart(shape, direction, tag, tile):
    p, a, b, n_out = operands(shape, direction, 5100)
    assert ops.halves_tile(p, direction, tag) == tile
    ref = reference(p, direction, a, b)
    guard = torch.full((n_out + 1024,), 7.0, device="cuda")
    got = launch(p, direction, tag, a, b, out=guard[:n_out])
    check(got, ref, products(p, direction), (shape, direction))
    assert torch.all(guard[n_out:] == 7.0)
    # (closer to 64 bits than additions in fp32: 3e-7 and more at these lengths)
    error = got.cpu().numpy().astype(np.float64).reshape(-1) - ref
    assert np.linalg.norm(error) <= 4e-7 * np.linalg.norm(ref.astype(np.float64))
    again = launch(p, direction, tag, a, b)
    assert torch.equal(again.view(torch.int32).reshape(-1),
                       got.view(torch.int32).reshape(-1))


@pytest.mark.parametrize("shape,direction,before", [
    ((17, 27, 27, 96, 256, 5, 1, True), F, 1.56e-7),   # parts inside a block of channels
    ((16, 16, 16, 192, 240, 5, 1, True), F, 1.58e-7),
    ((24, 39, 39, 32, 48, 7, 1, True), F, 1.77e-7),    # one block
    ((7, 36, 27, 128, 320, 4, 1, True), F, 1.43e-7),
    ((51, 26, 26, 204, 324, 3, 2, False), F, 1.42e-7),
    ((28, 18, 18, 176, 244, 3, 1, True), F, 1.25e-7),
    ((17, 39, 50, 48, 300, 3, 1, True), F, 9.0e-8),    # a short reduction
    ((13, 17, 22, 128, 480, 2, 1, True), F, 1.17e-7),  # eight waves' sums of their own
    ((40, 8, 10, 192, 208, 4, 1, True), I, 1.65e-7),
    ((16, 20, 26, 72, 512, 4, 1, True), I, 2.72e-7),
])
def test_error_is_that_of_the_kernel_before(shape, direction, before):
    """Against 64 bits in the 2-norm, normal values: no more than on the kernel that the
    layer has without room for the filter, whose error stands here (and a thirtieth:
    what the estimate of the parts is good for)."""
    p = ops.conv_params(*shape)
    rng = torch.Generator().manual_seed(5150)
    x_shape = (p.batch, p.in_rows, p.in_cols, p.channels)
    y_shape = (p.batch, p.out_rows, p.out_cols, p.features)
    k, s = p.window_rows, p.stride_rows
    w = torch.randn(k, k, p.channels, p.features, generator=rng).cuda()
    a = torch.randn(x_shape if direction == F else y_shape, generator=rng).cuda()
    if direction == F:
        a.relu_()
    rows = (p.out_rows - 1) * s + k
    cols = (p.out_cols - 1) * s + k
    whole = torch.zeros(p.batch, max(rows, p.pad_rows + p.in_rows),
                        max(cols, p.pad_cols + p.in_cols), p.channels,
                        dtype=torch.float64, device="cuda")
    inner = whole[:, p.pad_rows:p.pad_rows + p.in_rows,
                  p.pad_cols:p.pad_cols + p.in_cols]
    if direction == F:
        inner.copy_(a)
    y = torch.zeros(a.numel() // a.shape[-1] if direction == I else
                    p.batch * p.out_rows * p.out_cols, p.features,
                    dtype=torch.float64, device="cuda")
    for r in range(k):
        for c in range(k):
            taps = whole[:, r:r + (p.out_rows - 1) * s + 1:s,
                         c:c + (p.out_cols - 1) * s + 1:s]
            if direction == F:
                y += taps.reshape(-1, p.channels) @ w[r, c].double()
            else:
                taps += (a.double().reshape(-1, p.features) @
                         w[r, c].double().t().contiguous()).reshape(taps.shape)
    ref = (y if direction == F else inner).reshape(-1)
    algorithm = ops.default_algorithm(p, direction, DTYPE.F32)
    _, rec = ops.workspace_size(p, direction, algorithm, DTYPE.F32)
    got = ops.conv2d(a.reshape(-1), w.reshape(-1), p, direction, algorithm,
                     workspace=torch.empty(max(rec, 1), device="cuda"))
    error = (got.reshape(-1).double() - ref).norm() / ref.norm()
    assert error.item() <= 1.033 * before


@pytest.mark.parametrize("tag,shape", [
    (TILED, (9, 41, 43, 100, 68, 4, 1, False)),
    (TILED, (16, 27, 27, 96, 256, 5, 1, True)),   # in parts
    (WINO, (16, 28, 28, 96, 128, 3, 1, True))])
@pytest.mark.parametrize("relu", [False, True])
def test_bias_and_relu(tag, shape, relu):
    p, a, b, _ = operands(shape, F, 5200)
    assert ops.halves_tile(p, F, tag) is not None
    bias = uniform(np.random.default_rng(3), p.features)
    ref = reference(p, F, a, b).reshape(-1, p.features) + bias
    _, rec = ops.workspace_size(p, F, tag, DTYPE.F32)
    got = ops.conv2d_bias_act(dev(a), dev(b), dev(bias), p, tag, relu=relu,
                              workspace=torch.empty(rec, device="cuda"))
    check(got, np.maximum(ref, 0) if relu else ref, products(p, F) + 1, shape)


def compare(p, direction, tag, a, b, tolerance):
    """The error of every output against the sum of its products' magnitudes."""
    ref = reference(p, direction, a, b).astype(np.float64)
    size = reference(p, direction, np.abs(a), np.abs(b)).astype(np.float64)
    got = launch(p, direction, tag, a, b).cpu().numpy().reshape(-1)
    error = np.abs(got.astype(np.float64) - ref)
    # (and half the least fp32 number)
    assert np.all(error <= tolerance * size + 2.0**-149)


# Small: few enough that the reference in 64 bits is quick, but on this kernel.
SHAPE = (8, 28, 28, 96, 96, 4, 1, True)


@pytest.mark.parametrize("direction", [F, I])
@pytest.mark.parametrize("operand", [0, 1])
@pytest.mark.parametrize("exponents", [
    (0, -20), (0, -26), (0, -27), (0, -40), (0, -52), (0, -60), (0, -126),
    (40, -10), (100, -20), (-100, -126), (-120, -130), (100, 60)])
def test_values_beside_larger_ones(direction, operand, exponents):
    """Every other channel has the larger exponent and meets zeros, so that the
    outputs are sums of the smaller values alone: no bit of them may be missing.
    A binary16 pair holds 2^26 between them, a second pass 2^52, the fp32
    instruction the rest."""
    p, a, b, _ = operands(SHAPE, direction, 5300)
    assert ops.halves_tile(p, direction, TILED) is not None
    large, small = exponents
    depth = p.channels if direction == F else p.features
    odd = np.arange(depth) % 2 == 1
    scale = np.where(odd, 2.0**small, 2.0**large)
    # the reduction's channel is a's last dimension; b is [tap][c][f]
    va = a.reshape(-1, depth).astype(np.float64)
    vb = b.reshape(16, p.channels, p.features).astype(np.float64)
    by = odd[None, :, None] if direction == F else odd[None, None, :]
    if operand == 0:
        va, vb = va * scale, np.where(by, vb, 0)
    else:
        vb = vb * (scale[None, :, None] if direction == F else scale)
        va = np.where(odd, va, 0)
    a, b = va.astype(np.float32).reshape(-1), vb.astype(np.float32).reshape(-1)
    compare(p, direction, TILED, a, b, 2 * np.sqrt(16 * depth) * 2.0**-24)


@pytest.mark.parametrize("direction", [F, I])
@pytest.mark.parametrize("operand", [0, 1])
def test_exponents_that_change(direction, operand):
    """Blocks of channels, images and features of other sizes than their
    neighbours, zeros among them."""
    p, a, b, _ = operands(SHAPE, direction, 5400)
    rng = np.random.default_rng(9)
    depth = p.channels if direction == F else p.features
    if operand == 0:
        v = a.reshape(p.batch, -1, depth)
        v *= np.exp2(rng.integers(-12, 12, (p.batch, 1, depth // 32, 1)) *
                     np.ones((1, 1, 1, 32))).reshape(p.batch, 1, depth)
        v[1, :, :32] = 0
        v[2] = 0
    else:
        v = b.reshape(16, p.channels, p.features)
        v *= np.exp2(rng.integers(-12, 12, (1, p.channels // 32, 1,
                                            p.features // 32, 1)) *
                     np.ones((1, 1, 32, 1, 32))).reshape(1, p.channels, -1)
        v[:, :32, :32] = 0
        v[:, 64:] = 0
    compare(p, direction, TILED, a, b, 2 * np.sqrt(16 * depth) * 2.0**-24)


# Three blocks of 32 channels, sixteen and nine taps.
DROPS = [(F, TILED, (8, 28, 28, 96, 96, 4, 1, True)),
         (I, TILED, (8, 28, 28, 96, 96, 4, 1, True)),
         (F, WINO, (16, 28, 28, 96, 128, 3, 1, True)),
         (I, WINO, (16, 28, 28, 128, 96, 3, 1, True))]


@pytest.mark.parametrize("direction,tag,shape", DROPS)
@pytest.mark.parametrize("drops", [(5, 5), (14, 14), (20, 20), (30, 30),
                                   (30, 15), (15, 30)])
def test_sums_that_follow_both_operands_down(direction, tag, shape, drops):
    """The blocks of channels behind the first are smaller in both operands and hold
    values too small for their own exponents in both: the first one's sums are scaled
    up by all four powers of two together."""
    p, a, b, _ = operands(shape, direction, 5410)
    assert ops.halves_tile(p, direction, tag) is not None
    depth = p.channels if direction == F else p.features
    taps = p.window_rows * p.window_cols
    block = np.minimum(np.arange(depth) // 32, 1)
    # (the sums of the first block as large as they can be)
    va = np.where(block == 0, 0.99, a.reshape(-1, depth)) * np.exp2(-drops[0] * block)
    va[:, 40] *= 2.0**-28
    vb = np.moveaxis(b.reshape(taps, p.channels, p.features), 1 if direction == F else 2,
                     2)
    vb = np.where(block == 0, 0.99, vb) * np.exp2(-drops[1] * block)
    vb[..., 50] *= 2.0**-28
    vb = np.moveaxis(vb, 2, 1 if direction == F else 2)
    compare(p, direction, tag, va.astype(np.float32).reshape(-1),
            np.ascontiguousarray(vb, np.float32).reshape(-1),
            2 * np.sqrt(taps * depth) * 2.0**-24)


@pytest.mark.parametrize("direction,tag,shape", DROPS)
@pytest.mark.parametrize("zero", ["filter", "pixels"])
def test_exponents_behind_zeros(direction, tag, shape, zero):
    """The first block of one operand is zeros, so that the sums are zeros too where
    their exponent first changes, by up to 2^100 and more: magnitudes on both sides of
    where that power of two is none of fp32's."""
    p, a, b, _ = operands(shape, direction, 5420)
    assert ops.halves_tile(p, direction, tag) is not None
    depth = p.channels if direction == F else p.features
    taps = p.window_rows * p.window_cols
    va = a.reshape(-1, depth)
    vb = b.reshape(taps, p.channels, p.features)
    first = (slice(None), slice(0, 32)) if direction == F else \
        (slice(None), slice(None), slice(0, 32))
    if zero == "filter":
        vb[first] = 0
    else:
        va[:, :32] = 0
    for e in range(-54, -46):
        if zero == "filter":
            sa, sb = 2.0**-50, np.float64(2.0**e)
        else:
            # (the filter falls behind the zeros by what is missing to 2^128)
            sa, sb = 2.0**-85, np.full(vb.shape, 2.0**(e + 22))
            sb[first] = 1
        compare(p, direction, tag, (va * sa).astype(np.float32).reshape(-1),
                (vb * sb).astype(np.float32).reshape(-1),
                2 * np.sqrt(taps * depth) * 2.0**-24)


@pytest.mark.parametrize("direction", [F, I])
def test_results_beyond_fp32(direction):
    """Every output is one product of values far below the largest of their blocks,
    which are close to fp32's own: it overflows, and the sum is scaled by more than
    2^200 at the end."""
    p, a, b, _ = operands(SHAPE, direction, 5430)
    depth = p.channels if direction == F else p.features
    va = np.full((a.size // depth, depth), 2.0**127)
    va[:, 1::2] = 2.0**75
    # the tap that meets the output's own pixel
    vb = np.zeros((16, p.channels, p.features))
    if direction == F:
        vb[5, 33], vb[5, 33, ::32] = 2.0**75, 2.0**127
    else:
        vb[5, :, 33], vb[5, ::32, 33] = 2.0**75, 2.0**127
    got = launch(p, direction, TILED, va.astype(np.float32).reshape(-1),
                 vb.astype(np.float32).reshape(-1))
    assert torch.all(got == float("inf"))


@pytest.mark.parametrize("direction", [F, I])
@pytest.mark.parametrize("operand", [0, 1])
@pytest.mark.parametrize("value", [np.inf, np.nan, np.finfo(np.float32).max])
def test_infinities_stay_with_their_outputs(direction, operand, value):
    p, a, b, n_out = operands(SHAPE, direction, 5500)
    # (the largest finite value once: sums of several overflow on the way in fp32)
    (a, b)[operand][-1] = value
    if not np.isfinite(value):
        (a, b)[operand][:1] = value
        (a, b)[operand][-5:] = value
    ref = reference(p, direction, a, b)
    got = launch(p, direction, TILED, a, b).cpu().numpy().reshape(-1)
    ok = np.isfinite(ref)
    assert ok.any()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    n = products(p, direction)
    part = ok & (np.abs(ref) < 1e30)
    error = np.abs(got[part].astype(np.float64) - ref[part])
    assert error.max() <= 2 * n * 2.0**-24 * np.abs(ref[part]).max()


@pytest.mark.parametrize("direction,tag,shape", DROPS + [
    (F, TILED, (12, 37, 39, 128, 256, 3, 2, True)),     # stride 2
    (F, TILED, (6, 57, 61, 40, 36, 7, 1, True))])       # most windows at a border
@pytest.mark.parametrize("operand", [0, 1])
def test_many_infinities(direction, tag, shape, operand):
    """So many that every tile holds some; outputs whose windows lie partly in the
    padding are sums of the products that exist."""
    p, a, b, _ = operands(shape, direction, 5510)
    assert ops.halves_tile(p, direction, tag) is not None
    if operand == 0:
        a[::997] = np.inf
    else:
        # in the corner taps, of a few features' filters
        v = b.reshape(-1, p.channels, p.features)
        v[0, 3, ::9], v[-1, 1, ::7] = np.inf, np.nan
    ref = reference(p, direction, a, b)
    got = launch(p, direction, tag, a, b).cpu().numpy().reshape(-1)
    finite = np.isfinite(ref)
    assert finite.any() and not finite.all()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    n = products(p, direction)
    error = np.abs(got[finite].astype(np.float64) - ref[finite])
    assert error.max() <= 2 * np.sqrt(n) * n * 2.0**-24


def forward64(p, x, w):
    k = p.window_rows
    whole = torch.zeros(p.batch, p.out_rows + k - 1, p.out_cols + k - 1, p.channels,
                        dtype=torch.float64, device="cuda")
    whole[:, p.pad_rows:p.pad_rows + p.in_rows,
          p.pad_cols:p.pad_cols + p.in_cols] = x
    y = torch.zeros(p.batch * p.out_rows * p.out_cols, p.features,
                    dtype=torch.float64, device="cuda")
    for r in range(k):
        for c in range(k):
            taps = whole[:, r:r + p.out_rows, c:c + p.out_cols]
            y += taps.reshape(-1, p.channels) @ w[r, c].double()
    return y


@pytest.mark.parametrize("shape", [
    (2, 49, 55, 32, 68, 7, 1, True),     # 24 and 25 taps of one block
    (7, 29, 54, 64, 192, 4, 1, True),    # 6 and 10 of two
    (8, 29, 47, 48, 192, 5, 1, True)])   # 12 and 13, a block of half the channels
@pytest.mark.parametrize("kind", ["normal", "pixels", "filter", "both", "blocks",
                                  "zeros", "late"])
def test_parts_inside_blocks(shape, kind):
    """Sums that are taken among a block's taps, beside small values that pass a second
    time, exponents that change, zeros, and a block that ends on the fp32 instruction
    after parts of the tile are stored; with bias and ReLU behind the last part."""
    p = ops.conv_params(*shape)
    tag = ops.default_algorithm(p, F, DTYPE.F32)
    assert ops.halves_tile(p, F, tag) is not None
    rng = torch.Generator().manual_seed(5700)
    x = torch.randn(p.batch, p.in_rows, p.in_cols, p.channels, generator=rng)
    w = torch.randn(p.window_rows, p.window_rows, p.channels, p.features,
                    generator=rng) * 0.1

    def few(t):
        return torch.where(torch.rand(t.shape, generator=rng) < 1e-3, t * 2.0**-30, t)
    if kind in ("pixels", "both"):
        x = few(x)
    if kind in ("filter", "both"):
        w = few(w)
    if kind == "blocks":
        x[..., 32:] *= 2.0**-9
        w[:, :, 32:] *= 2.0**5
        x[0] *= 2.0**20
    if kind == "zeros":
        x[..., :32] = 0
        w[:, :, :, 5] = 0
    if kind == "late":
        x[0, 3, 4, -1] = 2.0**-100     # of the last block: beyond both exponents
        w[:, :, -1, 7] = 2.0**-90
    bias = torch.randn(p.features, generator=rng)
    x, w, bias = x.cuda(), w.cuda(), bias.cuda()
    ref, size = forward64(p, x, w), forward64(p, x.abs(), w.abs())
    _, rec = ops.workspace_size(p, F, tag, DTYPE.F32)
    ws = torch.empty(rec, device="cuda")
    n = products(p, F)
    got = ops.conv2d(x.reshape(-1), w.reshape(-1), p, F, tag, workspace=ws)
    error = (got.double().reshape(ref.shape) - ref).abs()
    assert torch.all(error <= 2 * np.sqrt(n) * 2.0**-24 * size + 2.0**-149)
    act = ops.conv2d_bias_act(x.reshape(-1), w.reshape(-1), bias, p, tag, relu=True,
                              workspace=ws).double().reshape(ref.shape)
    want = (got.double().reshape(ref.shape) + bias.double()).clamp_min(0)
    assert torch.all((act - want).abs() <= 2.0**-23 * want.abs() + 2.0**-149)


def test_prepared_filter_without_a_pack():
    """A prepared launch behind another tag than Winograd packs for itself."""
    p, a, b, _ = operands(SHAPE, F, 5600)
    _, rec = ops.workspace_size(p, F, TILED, DTYPE.F32)
    ws = torch.full((rec,), float("nan"), device="cuda")
    ops.conv2d_prepare_filter(dev(b), p, F, TILED, ws)
    got = ops.conv2d_prepared(dev(a), dev(b), p, F, TILED, ws)
    check(got, reference(p, F, a, b), products(p, F), "prepared")


def test_short_workspace_and_bad_arguments():
    """Without room for the filter such a launch runs on the kernels that need
    none."""
    p, a, b, _ = operands(SHAPE, F, 5700)
    ref = reference(p, F, a, b)
    for ws in (None, torch.empty(64, device="cuda")):
        got = ops.conv2d(dev(a), dev(b), p, F, TILED, workspace=ws)
        check(got, ref, products(p, F), "short workspace")
    fn = capi.lib().snn_hip_conv2d_halves_tile
    n = ctypes.c_int()
    assert fn(None, F, TILED, ctypes.byref(n), ctypes.byref(n)) == \
        capi.STATUS.INVALID_PARAMETER
    assert ops.halves_tile(p, DIRECTION.FILTER_BACKPROP, TILED) is None
    assert ops.halves_tile(p, F, ALGO.DIRECT) is None
