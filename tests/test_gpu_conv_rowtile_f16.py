"""Binary16 3x3 layers on the LDS-tile kernel: one tile of all 64 channels, two of 32
in turn, and one of 32 that is loaded again; whole rows per work-group and tiles that
start inside a row; one and two feature groups.  And wide images of few pixels, which
the rule leaves to the gathering kernel.

Bound: one rounding to binary16 and n fp32 additions.
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION, DTYPE
from test_gpu_conv_f16_shapes import assert_rounded_once, check_recorded
from test_gpu_parity import ORACLE_FN, dev, oracle_params, uniform

pytestmark = pytest.mark.gpu

# batch, rows, cols, source channels, produced channels, same
SHAPES = [
    (3, 37, 224, 64, 64, True),
    (1, 61, 300, 64, 64, True),
    (2, 47, 219, 64, 128, False),
    (1, 41, 224, 192, 64, True),
    (2, 29, 150, 64, 192, True),
    (9, 30, 31, 64, 64, True),
]


F, I = DIRECTION.FORWARD, DIRECTION.INPUT_BACKPROP
# ..., direction, form (ops.lds_form_f16)
FORMS = [
    ((7, 27, 39, 64, 192, True), F, 1),
    ((14, 11, 54, 64, 128, True), F, 1),
    ((8, 115, 53, 64, 64, False), I, 1),
    ((11, 39, 77, 64, 128, False), I, 1),
    ((13, 15, 49, 64, 128, True), F, 2),
    ((10, 17, 121, 128, 64, True), F, 2),
    ((1, 43, 119, 128, 256, True), F, 2),
    ((11, 65, 23, 128, 192, True), I, 2),
    ((13, 17, 75, 128, 256, True), I, 2),
    ((2, 129, 169, 64, 64, True), F, 3),
    ((3, 43, 107, 64, 256, True), F, 3),
    ((2, 69, 91, 128, 256, True), F, 3),
    ((5, 79, 185, 64, 64, True), I, 3),
    ((6, 63, 185, 128, 64, True), I, 3),
    ((5, 163, 78, 64, 128, False), I, 3),
]


@pytest.mark.parametrize(
    "shape,direction,form", FORMS,
    ids=["x".join(map(str, c[0])) + "fi"[c[1] == I] for c in FORMS])
def test_conv_rowtile_f16_forms(shape, direction, form):
    batch, rows, cols, source, produced, same = shape
    channels, features = ((source, produced) if direction == F
                          else (produced, source))
    assert ops.lds_form_f16(
        ops.conv_params(batch, rows, cols, channels, features, 3, 1, same),
        direction) == form
    check(shape, direction)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("direction", [F, I])
def test_conv_rowtile_f16(shape, direction):
    check(shape, direction)


def check(shape, direction):
    batch, rows, cols, source, produced, same = shape
    channels, features = ((source, produced) if direction == DIRECTION.FORWARD
                          else (produced, source))
    p = ops.conv_params(batch, rows, cols, channels, features, 3, 1, same)
    rng = np.random.default_rng(9100 + rows + cols)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a = uniform(rng, n_a).astype(np.float16)
    b = uniform(rng, n_b).astype(np.float16)
    ref = ORACLE_FN[direction](a.astype(np.float32), b.astype(np.float32),
                               oracle_params(p, features), acc64=True)
    _, rec = ops.workspace_size(p, direction, ALGO.IM2COL, DTYPE.F16)
    block = torch.full((rec + 4096,), 7.0, dtype=torch.float16, device="cuda")
    guard = torch.full((n_out + 4096,), 7.0, dtype=torch.float16, device="cuda")
    got = ops.conv2d(dev(a, torch.float16), dev(b, torch.float16), p, direction,
                     ALGO.IM2COL, workspace=block[:rec], out=guard[:n_out])
    assert_rounded_once(got.float().cpu().numpy(), ref, 9 * source,
                        (shape, direction))
    assert torch.all(guard[n_out:] == 7.0)
    assert torch.all(block[rec:] == 7.0)


@pytest.mark.parametrize("shape", [c[0] for c in FORMS if c[1] == I][:4],
                         ids=lambda s: "x".join(map(str, s)))
def test_input_gradient_recorded_without_a_workspace(shape):
    """Kernels only: the gathering kernel reads the filter in place."""
    batch, rows, cols, source, produced, same = shape
    p = ops.conv_params(batch, rows, cols, produced, source, 3, 1, same)
    n_a, n_b, n_out = ops.conv_sizes(p, I)
    a = torch.empty(n_a, dtype=torch.float16, device="cuda")
    b = torch.empty(n_b, dtype=torch.float16, device="cuda")

    def refill(seed):
        rng = np.random.default_rng(seed)
        a.copy_(dev(uniform(rng, n_a), torch.float16))
        b.copy_(dev(uniform(rng, n_b), torch.float16))

    refill(0)
    check_recorded(lambda out: ops.conv2d(a, b, p, I, ALGO.IM2COL, out=out),
                   refill, 9 * source, shape)
