"""fp32 filter gradients whose operands are taken apart into two binary16 values: ragged
channels and features, segments of rows, bands, several bands a task, several tasks and
splits; exponents that change between tasks, values too small for them, zeros,
infinities and NaNs.

Bound: a sum of at most n products in fp32, an operand off by at most 2^-23 of itself:
(n + 8) 2^-24 of the sum of the products' magnitudes.
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE

pytestmark = pytest.mark.gpu

W = DIRECTION.FILTER_BACKPROP
TILED, WINO = ALGO.IM2COL, ALGO.WINOGRAD
# batch, rows, cols, channels, features, window, same; tag; partial filters
CASES = [
    ((32, 28, 28, 128, 128, 3, True), WINO, 32),
    ((8, 56, 56, 64, 64, 3, True), WINO, 75),
    ((22, 7, 7, 96, 64, 3, True), WINO, 11),       # several bands a task
    ((11, 19, 130, 36, 100, 3, True), TILED, 53),   # segments
    ((43, 21, 21, 32, 528, 3, False), TILED, 26),
    ((1, 14, 14, 16, 16, 3, True), TILED, 7),      # the smallest counts
    ((5, 33, 20, 20, 68, 3, True), TILED, 45),
    ((17, 27, 27, 96, 256, 5, True), TILED, 17),
    ((6, 97, 40, 56, 16, 5, False), TILED, 47),
    ((70, 15, 15, 76, 144, 5, False), TILED, 23),
]
IDS = ["x".join(map(str, c[0])) for c in CASES]


def operands(shape, seed):
    n, h, w, c, f, k, same = shape
    p = ops.conv_params(n, h, w, c, f, k, 1, same)
    rng = torch.Generator().manual_seed(seed)
    x = torch.randn(n, h, w, c, generator=rng).relu_()
    dy = torch.randn(n, p.out_rows, p.out_cols, f, generator=rng) * 0.1
    return p, x, dy


def reference(p, x, dy):
    """dW and the sums of the products' magnitudes, in 64 bits."""
    k = p.window_rows
    x, dy = x.cuda().double(), dy.cuda().double().reshape(-1, p.features)
    rows = p.out_rows + k - 1 - p.in_rows - p.pad_rows
    cols = p.out_cols + k - 1 - p.in_cols - p.pad_cols
    x = torch.nn.functional.pad(x, (0, 0, p.pad_cols, cols, p.pad_rows, rows))
    taps = [x[:, r:r + p.out_rows, s:s + p.out_cols].reshape(-1, p.channels)
            for r in range(k) for s in range(k)]
    return (torch.stack([t.t() @ dy for t in taps]),
            torch.stack([t.abs().t() @ dy.abs() for t in taps]))


def launch(p, tag, x, dy, room=None):
    _, rec = ops.workspace_size(p, W, tag, DTYPE.F32)
    room = rec if room is None else room
    ws = torch.full((room + 1024,), 7.0, device="cuda")
    n_out = p.window_rows * p.window_cols * p.channels * p.features
    out = torch.full((n_out + 1024,), 7.0, device="cuda")
    ops.conv2d(x.cuda().reshape(-1), dy.cuda().reshape(-1), p, W, tag,
               workspace=ws[:room], out=out[:n_out])
    assert torch.all(ws[room:] == 7.0) and torch.all(out[n_out:] == 7.0)
    return out[:n_out].reshape(-1, p.channels, p.features)


def check(p, got, x, dy, what):
    ref, norm = reference(p, x, dy)
    pixels = p.batch * p.out_rows * p.out_cols
    over = (got.double() - ref).abs() - (pixels + 8) * 2.0 ** -24 * norm
    assert torch.all(over <= 0), (what, over.max().item())
    return ((got.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("shape,tag,partials", CASES, ids=IDS)
def test_taken_apart(shape, tag, partials):
    p, x, dy = operands(shape, 3)
    assert ops.filter_halves_partials(p, tag) == partials
    got = launch(p, tag, x, dy)
    # (sums in fp32 alone are off by as much from 300 pixels on)
    assert check(p, got, x, dy, shape) <= 4e-7
    again = launch(p, tag, x, dy)
    assert torch.equal(got.view(torch.int32), again.view(torch.int32))


@pytest.mark.parametrize("shape,before", [
    ((35, 8, 7, 652, 32, 5, True), 1.403e-7),
    ((36, 8, 8, 160, 96, 5, True), 1.283e-7),
    ((40, 12, 12, 368, 48, 5, True), 1.625e-7),
    ((9, 13, 13, 156, 544, 5, True), 1.702e-7),
    ((5, 20, 15, 160, 208, 5, True), 1.324e-7),
    ((49, 20, 26, 64, 16, 3, False), 1.727e-7),
    ((17, 27, 27, 96, 256, 5, True), 2.300e-7),
])
def test_error_is_that_of_the_kernel_before(shape, before):
    """Against 64 bits in the 2-norm: no more than on the kernel that loads its operands
    into registers, whose error stands here (and a fiftieth: other normal values)."""
    p, x, dy = operands(shape, 11)
    algorithm = ops.default_algorithm(p, W, DTYPE.F32)
    ref, _ = reference(p, x, dy)
    got = launch(p, algorithm, x, dy).double()
    assert ((got - ref).norm() / ref.norm()).item() <= 1.02 * before


@pytest.mark.parametrize("shape,tag", [
    ((16, 28, 28, 64, 64, 3, True), WINO), ((43, 21, 21, 32, 68, 3, False), TILED),
    ((17, 27, 27, 96, 64, 5, True), TILED)])
@pytest.mark.parametrize("kind", [
    "images", "pixels", "small_x", "small_both", "zeros", "channels", "tiny"])
def test_ranges(shape, tag, kind):
    """Magnitudes that differ between tasks, within one, and by more than the second
    exponent holds."""
    p, x, dy = operands(shape, 5)
    assert ops.filter_halves_partials(p, tag)
    rng = torch.Generator().manual_seed(6)

    def scales(like, most):
        return torch.exp2(-torch.randint(0, most, like, generator=rng).float())
    if kind == "images":
        x *= scales((p.batch, 1, 1, 1), 60)
        dy *= scales((p.batch, 1, 1, 1), 60) * 2.0 ** 30
    elif kind == "pixels":
        dy *= scales(dy.shape[:3] + (1,), 45)
    elif kind == "small_x":
        x *= scales(x.shape, 40)
    elif kind == "small_both":
        x *= scales(x.shape, 34)
        dy *= scales(dy.shape, 34)
    elif kind == "zeros":
        x[: p.batch // 2] = 0
        dy[p.batch // 4:] = 0
        x[-1], dy[-1] = 1e-6, 3e5
    elif kind == "channels":
        x[..., 3] *= 2.0 ** -70
        dy[..., 5] *= 2.0 ** 50
    else:
        x *= 2.0 ** -100
        dy *= 2.0 ** -30
    got = launch(p, tag, x, dy)
    ref, norm = reference(p, x, dy)
    pixels = p.batch * p.out_rows * p.out_cols
    # (2^-126: where results below the normal range are rounded)
    bound = (pixels + 8) * 2.0 ** -24 * norm + 2.0 ** -126
    over = (got.double() - ref).abs() - bound
    assert torch.all(over <= 0), over.max().item()


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3e38])
@pytest.mark.parametrize("at", ["x", "dy"])
def test_not_finite(value, at):
    """They reach the sums that they belong to and no others; an input pixel beside the
    last column meets padding's dY nowhere."""
    p, x, dy = operands((8, 28, 28, 64, 64, 3, True), 7)
    dy += 0.5  # (no zeros beside an infinity)
    if at == "x":
        x[1, 27, 27, 17] = value
    else:
        dy[1, 13, 13, 17] = value
    got = launch(p, WINO, x, dy)
    ref, _ = reference(p, x, dy)
    hit = ~torch.isfinite(ref.float()) | (ref.abs() > 1e30)
    taps = 4 if at == "x" else 9
    assert hit.any() and hit.sum().item() <= taps * 64
    if value == value and abs(value) > 3.4e38 or value != value:
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
    rest = ~hit
    assert torch.allclose(got[rest].double(), ref[rest], rtol=1e-4, atol=1e-3)


def test_results_beyond_fp32():
    """Every element is one product of values far below the largest of their task,
    which are close to fp32's own: it overflows, and the sum is scaled by more than
    2^200 at the end."""
    p, x, dy = operands((16, 28, 28, 64, 64, 3, True), 8)
    x[:], dy[:] = 2.0 ** 76, 0
    x[..., 0] = 2.0 ** 127
    dy[0, 13, 13] = 2.0 ** 76
    dy[0, 13, 13, 0] = 2.0 ** 127
    assert torch.all(launch(p, WINO, x, dy) == float("inf"))


def test_short_workspace():
    """Without room for the partial filters: a temporary behind the Im2col tag, the
    Winograd kernel behind its own."""
    p, x, dy = operands((17, 27, 27, 96, 256, 5, True), 9)
    got = launch(p, TILED, x, dy, room=4096)
    assert torch.equal(got, launch(p, TILED, x, dy))
    q, x, dy = operands((32, 28, 28, 128, 128, 3, True), 9)
    need, rec = ops.workspace_size(q, W, WINO, DTYPE.F32)
    assert need < rec
    check(q, launch(q, WINO, x, dy, room=need), x, dy, "required")
