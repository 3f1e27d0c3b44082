"""Conv backward weight without LDS staging (conv_wgrad_direct.hip): edges of its 16 / 32 / 64-channel
and 32-element tiles, of an image's 16-pixel steps, of the waves' and slices' runs of steps; strides,
padding, 1x1 layers; with and without a caller workspace.  Against fp64 within twice the error of the
reference's route (plus one rounding for short sums)."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import F32_FLOOR, dev, host, normal, require_gpu, say

pytestmark = pytest.mark.gpu

# batch, IC, OC, H, W, KH, KW, stride, padding
GEOMS = [
    (1, 1, 1, 1, 1, 1, 1, (1, 1), (0, 0)),        # one product
    (1, 3, 16, 4, 4, 3, 3, (1, 1), (1, 1)),       # one whole step, three waves without work
    (3, 5, 17, 5, 7, 3, 3, (1, 1), (1, 1)),       # 35 pixels: short last steps
    (2, 4, 33, 9, 9, 5, 3, (2, 1), (2, 0)),
    (5, 33, 65, 7, 7, 3, 3, (1, 1), (2, 2)),      # padding as wide as the filter
    (4, 7, 48, 30, 17, 7, 7, (2, 3), (3, 3)),     # slices
    (1, 60, 24, 33, 1, 3, 1, (3, 1), (1, 0)),     # one column
    (9, 31, 130, 1, 1, 1, 1, (1, 1), (0, 0)),     # 1x1 on one pixel
    (6, 65, 96, 13, 11, 1, 1, (1, 1), (0, 0)),    # 1x1 with short steps
    (16, 64, 64, 28, 28, 1, 1, (1, 1), (0, 0)),   # 1x1, slices of whole steps
    (2, 70, 40, 12, 12, 1, 1, (2, 2), (0, 0)),
    (2, 8, 20, 16, 16, 3, 3, (1, 1), (1, 1)),     # rows of 16
]


@pytest.mark.parametrize("g", GEOMS)
def test_weight_grad(g):
    require_gpu()
    import torch
    import cudeep_amd.ops as ops
    B, IC, OC, H, W, KH, KW, stride, pad = g
    rng = np.random.default_rng(sum(g[:7]))
    oh, ow = (H + 2 * pad[0] - KH) // stride[0] + 1, (W + 2 * pad[1] - KW) // stride[1] + 1
    x, dy = normal(rng, (B, IC, H, W)), normal(rng, (B, OC, oh, ow))
    shape = (OC, IC, KH, KW)
    d64 = oracle.conv2d_backward_weight64(dy, x, shape, stride, pad)
    ref = oracle.conv2d_backward_weight_ref(dy, x, shape, stride, pad)
    say("wgrad direct", g)
    dw = ops.conv2d_backward_weight(dev(dy), dev(x), shape, stride, pad)
    assert oracle.rel_fro(host(dw), d64) <= 2 * oracle.rel_fro(ref, d64) + F32_FLOOR
    n = ops.conv2d_backward_weight_workspace_bytes(x.shape, shape, stride, pad)
    ws = torch.full((n // 4 + 1,), float("nan"), device="cuda")
    again = ops.conv2d_backward_weight(dev(dy), dev(x), shape, stride, pad, workspace=ws)
    assert torch.equal(dw, again)
