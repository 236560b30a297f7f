"""Depthwise 3x3 filter gradients: the sum of the work-groups' partial filters,
over few and many work-groups, filters that are no multiple of the 16 vectors
of a summing work-group, and, in fp32, both ways the sums take (atomics while
they are few).  The gradient overwrites whatever its buffer held, eagerly and
on every replay of a captured graph.

Bound: n fp32 additions, and in binary16 one rounding on top.
"""
import numpy as np
import pytest
import torch

from portdnn_amd import ops
from portdnn_amd.capi import DIRECTION

pytestmark = pytest.mark.gpu

# batch, rows, cols, channels, stride
SHAPES = [(9, 28, 28, 40, 1),      # few work-groups; 90 vectors
          (40, 56, 56, 4, 1),      # one vector of channels
          (5, 115, 113, 36, 2),    # ragged at stride 2
          (16, 112, 112, 32, 1),   # atomics in fp32 no longer
          (24, 57, 55, 260, 1),    # 585 vectors, ragged lanes of channels
          (70, 14, 14, 512, 1),    # four columns of work-groups
          (33, 14, 15, 512, 2)]


def reference(x, dy, p, stride):
    x = np.pad(x.astype(np.float64),
               ((0, 0), (p.pad_rows, 2 + stride), (p.pad_cols, 2 + stride),
                (0, 0)))
    dy = dy.astype(np.float64)
    dw = np.zeros((3, 3, x.shape[3]))
    size = np.zeros_like(dw)
    for r in range(3):
        for c in range(3):
            part = x[:, r:r + stride * p.out_rows:stride,
                     c:c + stride * p.out_cols:stride]
            dw[r, c] = np.einsum("bijc,bijc->c", part, dy)
            size[r, c] = np.einsum("bijc,bijc->c", np.abs(part), np.abs(dy))
    return dw, size


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16],
                         ids=["f32", "f16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_partial_filters_add_up(shape, dtype):
    batch, rows, cols, channels, stride = shape
    p = ops.depthwise_params(batch, rows, cols, channels, 1, 3, stride, True)
    rng = np.random.default_rng(sum(shape))
    kind = np.float32 if dtype == torch.float32 else np.float16
    x = rng.uniform(-1, 1, (batch, rows, cols, channels)).astype(kind)
    dy = rng.uniform(-1, 1, (batch, p.out_rows, p.out_cols,
                             channels)).astype(kind)
    dx, ddy = torch.from_numpy(x).cuda(), torch.from_numpy(dy).cuda()
    dw = torch.full((3, 3, channels), float("nan"), dtype=dtype, device="cuda")

    def run():
        ops.depthwise_conv2d(dx, ddy, p, DIRECTION.FILTER_BACKPROP, out=dw)

    want, size = reference(x, dy, p, stride)
    n = batch * p.out_rows * p.out_cols
    # fp32 products and additions in any order lose at most n roundings of the
    # sum of the magnitudes
    bound = n * 2.0**-24 * size
    if dtype == torch.float16:
        bound = bound + 2.0**-11 * np.abs(want) + 2.0**-25

    def check(what):
        err = np.abs(dw.double().cpu().numpy() - want)
        assert np.all(err <= bound), (what, err.max())

    run()
    check("eager")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for replay in range(3):
        dw.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        check(("replay", replay))
        run()
        check(("eager after replay", replay))
