"""fp32 Winograd launches of few units of work, which run on the kernels behind the
Tiled tag where those are faster, with the filter transformed ahead as well where
nothing is written over the transformed filter."""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import ALGO, DIRECTION
from test_gpu_parity import (ORACLE_FN, assert_close, dev, oracle_params,
                             uniform)

pytestmark = pytest.mark.gpu

# batch, rows, cols, channels, features, same
SHAPES = [
    (1, 56, 56, 64, 64, True),    # the kernel for small layers
    (3, 13, 11, 16, 64, True),    # one chunk of 16 channels
    (2, 9, 10, 128, 32, False),   # eight chunks
    (1, 7, 7, 512, 512, True),    # split channel range
    (5, 6, 5, 48, 96, True),      # a line of the rule on each side
    (5, 38, 28, 64, 96, True),
]


@pytest.mark.parametrize("direction", [DIRECTION.FORWARD,
                                       DIRECTION.INPUT_BACKPROP])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_winograd_few_units(shape, direction):
    batch, rows, cols, channels, features, same = shape
    if direction == DIRECTION.INPUT_BACKPROP:
        channels, features = features, channels
    p = ops.conv_params(batch, rows, cols, channels, features, 3, 1, same)
    rng = np.random.default_rng(8100 + rows)
    n_a, n_b, _ = ops.conv_sizes(p, direction)
    a, b = uniform(rng, n_a), uniform(rng, n_b)
    ref = np.asarray(ORACLE_FN[direction](
        a, b, oracle_params(p, features), acc64=True)).reshape(-1)
    da, db = dev(a), dev(b)
    _, rec = ops.workspace_size(p, direction, ALGO.WINOGRAD)
    ws = torch.empty(rec, dtype=torch.float32, device="cuda")
    plain = ops.conv2d(da, db, p, direction, ALGO.WINOGRAD, workspace=ws)
    assert_close(plain.cpu().numpy(), ref, (shape, direction))
    ops.conv2d_prepare_filter(db, p, direction, ALGO.WINOGRAD, ws)
    for _ in range(2):
        got = ops.conv2d_prepared(da, db, p, direction, ALGO.WINOGRAD, ws)
        assert_close(got.cpu().numpy(), ref, (shape, direction, "prepared"))
    ws.fill_(float("nan"))
    ops.conv2d_prepare_filter(db, p, direction, ALGO.WINOGRAD, ws)
    ops.conv2d_prepared(da, db, p, direction, ALGO.WINOGRAD, ws)
    unaligned = torch.empty(n_b + 1, dtype=torch.float32, device="cuda")[1:]
    unaligned.copy_(db)
    got = ops.conv2d_prepared(da, unaligned, p, direction, ALGO.WINOGRAD, ws)
    assert_close(got.cpu().numpy(), ref, (shape, direction, "unaligned"))
    same_bits = [ops.conv2d_deterministic(da, db, p, direction, ALGO.WINOGRAD,
                                          ws) for _ in range(2)]
    assert torch.equal(*same_bits)
    assert_close(same_bits[0].cpu().numpy(), ref, (shape, "deterministic"))
    if direction == DIRECTION.FORWARD:
        bias = uniform(rng, features)
        want = np.maximum(ref.reshape(-1, features) + bias, 0).reshape(-1)
        got = ops.conv2d_bias_act(da, db, dev(bias), p, ALGO.WINOGRAD,
                                  relu=True, workspace=ws)
        assert_close(got.cpu().numpy(), want, (shape, "bias"))


@pytest.mark.parametrize("direction", [DIRECTION.FORWARD,
                                       DIRECTION.INPUT_BACKPROP])
@pytest.mark.parametrize("shape", SHAPES + [
    (1, 56, 56, 96, 96, True),    # tiles that would share a reduction ...
    (2, 14, 14, 160, 96, True),   # ... and a split channel range
    (3, 14, 14, 64, 64, True),
    (9, 20, 42, 16, 736, True),
    (16, 28, 28, 96, 128, True),  # its filter is taken apart into binary16 values
], ids=lambda s: "x".join(map(str, s)))
def test_prepared_workspace_is_only_read(shape, direction):
    """What a filter was transformed to survives every prepared launch, aligned or
    not, so that launches on other streams can read it meanwhile; and a layer whose
    channel range is not split gives the bits of the one-call launch."""
    batch, rows, cols, channels, features, same = shape
    p = ops.conv_params(batch, rows, cols, *(
        (channels, features) if direction == DIRECTION.FORWARD else
        (features, channels)), 3, 1, same)
    assert (ops.halves_tile(p, direction, ALGO.WINOGRAD) is not None) == (batch == 16)
    rng = np.random.default_rng(8200 + rows)
    n_a, n_b, n_out = ops.conv_sizes(p, direction)
    a, b = uniform(rng, n_a), uniform(rng, n_b)
    ref = np.asarray(ORACLE_FN[direction](
        a, b, oracle_params(p, p.features), acc64=True)).reshape(-1)
    da, db = dev(a), dev(b)

    def moved(t):
        u = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:]
        u.copy_(t.reshape(-1))
        return u

    _, rec = ops.workspace_size(p, direction, ALGO.WINOGRAD)
    ws = torch.full((rec,), 7.0, device="cuda")
    ops.conv2d_prepare_filter(db, p, direction, ALGO.WINOGRAD, ws)
    held = ws.clone()
    out = torch.empty(n_out + 4, device="cuda")
    for x, w, y in ((da, db, out[:n_out]), (moved(da), db, out[:n_out]),
                    (da, moved(db), out[:n_out]), (da, db, out[1:n_out + 1])):
        y.fill_(float("nan"))
        ops.conv2d_prepared(x, w, p, direction, ALGO.WINOGRAD, ws, out=y)
        assert_close(y.cpu().numpy(), ref, (shape, direction))
        assert torch.equal(ws.view(torch.int32), held.view(torch.int32))
    if channels < 128:
        two = ops.conv2d_prepared(da, db, p, direction, ALGO.WINOGRAD, ws)
        one = ops.conv2d(da, db, p, direction, ALGO.WINOGRAD, workspace=ws)
        assert torch.equal(one.view(torch.int32), two.view(torch.int32))


@pytest.mark.parametrize("shape,direction", [
    ((32, 36, 9, 16, 640), DIRECTION.FORWARD),
    ((32, 23, 77, 16, 128), DIRECTION.FORWARD),
    ((32, 9, 54, 16, 768), DIRECTION.INPUT_BACKPROP),
    ((16, 28, 28, 32, 128), DIRECTION.INPUT_BACKPROP),
    ((12, 33, 31, 48, 96), DIRECTION.FORWARD)],
    ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else str(s))
def test_prepared_filter_takes_sixteen_values(shape, direction):
    """A prepared launch reads the first 16 * C * K elements of its workspace and no
    others; whatever the filter was turned to fits there."""
    batch, rows, cols, channels, features = shape
    p = ops.conv_params(batch, rows, cols, *(
        (channels, features) if direction == DIRECTION.FORWARD else
        (features, channels)), 3, 1, True)
    rng = np.random.default_rng(8300 + rows)
    n_a, n_b, _ = ops.conv_sizes(p, direction)
    a, b = uniform(rng, n_a), uniform(rng, n_b)
    ref = np.asarray(ORACLE_FN[direction](
        a, b, oracle_params(p, p.features), acc64=True)).reshape(-1)
    _, rec = ops.workspace_size(p, direction, ALGO.WINOGRAD)
    ws = torch.empty(rec, device="cuda")
    ops.conv2d_prepare_filter(dev(b), p, direction, ALGO.WINOGRAD, ws)
    ws[16 * channels * features:] = float("nan")
    got = ops.conv2d_prepared(dev(a), dev(b), p, direction, ALGO.WINOGRAD, ws)
    assert_close(got.cpu().numpy(), ref, (shape, direction))
