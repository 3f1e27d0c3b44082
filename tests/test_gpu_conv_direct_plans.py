"""Every form of the convolution whose waves gather their own operands (conv_direct.hip): 16, 32 and
64 channels per wave, k split over a workgroup's waves and not, each with a ragged last channel
tile, pixels past the last tile and more k than one table.  Forward, and stride-1 backward data.
Against fp64 within twice the error of the reference's own route (plus one rounding)."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import F32_FLOOR, dev, host, normal, require_gpu, say
from tests.routes import conv_kernel

pytestmark = pytest.mark.gpu


def plan(N, OC, K):
    """conv_direct.hip's plan_of(): channels per wave in sixteens, k split."""
    up = lambda a, b: -(-a // b)
    fm = 1 if OC <= 16 else 4
    if fm == 4 and (up(OC, 32) * 32 * 115 < up(OC, 64) * 64 * 100 or up(N, 32) * up(OC, 64) < 150):
        fm = 2
    if fm == 2 and up(N, 32) * up(OC, 32) < 64:
        fm = 1
    return fm, K >= 128 and up(N, 32) * up(OC, 16 * fm) < 4096


# batch, IC, OC, H, W, KH, KW, stride, padding; the plan
FORWARD = [
    ((4, 128, 125, 28, 28, 3, 3, (1, 1), (1, 1)), (4, True)),     # 1152 k: two tables
    ((3, 15, 190, 41, 39, 3, 3, (1, 1), (2, 0)), (4, True)),      # 135 k, one-pixel tail
    ((5, 100, 121, 57, 55, 1, 1, (2, 2), (0, 0)), (4, False)),
    ((2, 120, 72, 21, 23, 3, 3, (1, 1), (1, 1)), (2, True)),
    ((4, 12, 94, 31, 33, 3, 3, (2, 2), (1, 1)), (2, False)),
    ((1, 118, 33, 9, 11, 3, 3, (1, 1), (1, 1)), (1, True)),
    ((2, 5, 15, 61, 60, 3, 5, (1, 2), (1, 2)), (1, False)),
]
DATA = [
    ((4, 125, 128, 28, 28, 3, 3, (1, 1), (1, 1)), (4, True)),
    ((3, 190, 15, 41, 39, 3, 3, (1, 1), (2, 0)), (4, True)),
    ((2, 72, 120, 21, 23, 3, 3, (1, 1), (1, 1)), (2, True)),
    ((4, 94, 12, 15, 17, 3, 3, (1, 1), (1, 1)), (2, False)),
    ((1, 33, 118, 9, 11, 3, 3, (1, 1), (1, 1)), (1, True)),
    ((2, 15, 5, 61, 30, 3, 5, (1, 1), (1, 2)), (1, False)),
]


def test_all_plans_are_covered():
    assert {p for _, p in FORWARD} == {(f, s) for f in (1, 2, 4) for s in (False, True)}
    assert {p for _, p in DATA} == {p for _, p in FORWARD} - {(4, False)}   # (1x1 layers are products)


@pytest.mark.parametrize("g,want", FORWARD)
def test_forward(g, want):
    require_gpu()
    import cudeep_amd.ops as ops
    B, IC, OC, H, W, KH, KW, stride, pad = g
    oh, ow = (H + 2 * pad[0] - KH) // stride[0] + 1, (W + 2 * pad[1] - KW) // stride[1] + 1
    assert conv_kernel("implicit", *g) == "direct" and plan(B * oh * ow, OC, IC * KH * KW) == want
    rng = np.random.default_rng(sum(g[:7]))
    x, w = normal(rng, (B, IC, H, W)), normal(rng, (OC, IC, KH, KW), (2.0 / (IC * KH * KW)) ** 0.5)
    b = normal(rng, (OC,))
    say("conv direct plans forward", g, want)
    y = host(ops.conv2d_implicit(dev(x), dev(w), dev(b), stride, pad))
    y64 = oracle.conv2d_direct64(x, w, b, stride, pad)
    ref = oracle.conv2d_ref_implicit(x, w, b, stride, pad)
    assert oracle.rel_fro(y, y64) <= 2 * oracle.rel_fro(ref, y64) + F32_FLOOR


@pytest.mark.parametrize("g,want", DATA)
def test_backward_data(g, want):
    require_gpu()
    import cudeep_amd.ops as ops
    B, IC, OC, H, W, KH, KW, stride, pad = g
    assert conv_kernel("data", *g) == "direct" and plan(B * H * W, IC, OC * KH * KW) == want
    rng = np.random.default_rng(sum(g[:7]) + 1)
    w = normal(rng, (OC, IC, KH, KW), (2.0 / (IC * KH * KW)) ** 0.5)
    dy = normal(rng, (B, OC, H + 2 * pad[0] - KH + 1, W + 2 * pad[1] - KW + 1))
    d64 = oracle.conv2d_backward_data64(dy, w, (B, IC, H, W), stride, pad)
    ref = oracle.conv2d_backward_data_ref(dy, w, (B, IC, H, W), stride, pad)
    say("conv direct plans backward data", g, want)
    dx = host(ops.conv2d_backward_data(dev(dy), dev(w), (B, IC, H, W), stride, pad))
    assert oracle.rel_fro(dx, d64) <= 2 * oracle.rel_fro(ref, d64) + F32_FLOOR
