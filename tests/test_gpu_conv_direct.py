"""Convolutions whose waves gather their own operands (conv_direct.hip) and 1x1 layers as plain
products: edges of the 32-pixel and 16-channel tiles, of the 16-k steps, of the 1024-k tables and of
the four k runs, padding and strides (32- and 64-channel waves: test_gpu_conv_direct_plans.py).  Forward and stride-1 backward data against
fp64 within twice the error of the reference's own route (plus one rounding for short sums)."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import F32_FLOOR, dev, host, normal, require_gpu, say

pytestmark = pytest.mark.gpu

# batch, IC, OC, H, W, KH, KW, stride, padding
GEOMS = [
    (1, 1, 1, 9, 9, 3, 3, (1, 1), (1, 1)),          # one channel either way, k = 9
    (1, 3, 17, 11, 13, 5, 3, (1, 1), (2, 1)),       # k = 45, 17 channels
    (2, 9, 16, 7, 7, 5, 3, (2, 1), (2, 0)),         # k = 135: split, one-pixel tail
    (1, 16, 33, 8, 4, 3, 3, (1, 1), (2, 2)),        # 32 + 1 channels; padding as wide as the filter
    (3, 15, 48, 6, 11, 3, 3, (1, 2), (0, 1)),
    (1, 114, 20, 5, 6, 3, 3, (1, 1), (1, 1)),       # k = 1026: two tables, the second of 2 k
    (1, 21, 72, 14, 14, 7, 7, (1, 1), (3, 3)),      # k = 1029, 49 taps
    (2, 30, 65, 12, 10, 7, 9, (1, 1), (3, 4)),      # 63 taps, all a mask holds
    (1, 25, 10, 20, 20, 8, 8, (1, 1), (0, 0)),      # 64 taps: another route
    (2, 70, 130, 9, 7, 1, 1, (2, 2), (0, 0)),       # 1x1 with stride
    (1, 6, 7, 33, 1, 3, 1, (3, 1), (1, 0)),         # one column
]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def ops():
    import cudeep_amd.ops as o
    return o


@pytest.mark.parametrize("g", GEOMS)
def test_forward(g):
    B, IC, OC, H, W, KH, KW, stride, pad = g
    rng = np.random.default_rng(sum(g[:7]))
    x, w = normal(rng, (B, IC, H, W)), normal(rng, (OC, IC, KH, KW), (2.0 / (IC * KH * KW)) ** 0.5)
    b = normal(rng, (OC,))
    y64 = oracle.conv2d_direct64(x, w, b, stride, pad)
    bar = 2 * oracle.rel_fro(oracle.conv2d_ref_implicit(x, w, b, stride, pad), y64) + F32_FLOOR
    say("conv direct forward", g)
    for y in (ops().conv2d_implicit(dev(x), dev(w), dev(b), stride, pad),
              ops().conv2d_forward(dev(x), dev(w), dev(b), stride, pad)):
        assert oracle.rel_fro(host(y), y64) <= bar


@pytest.mark.parametrize("g", [g for g in GEOMS if g[7] == (1, 1)])
def test_backward_data(g):
    B, IC, OC, H, W, KH, KW, stride, pad = g
    rng = np.random.default_rng(sum(g[:7]) + 1)
    w = normal(rng, (OC, IC, KH, KW), (2.0 / (IC * KH * KW)) ** 0.5)
    dy = normal(rng, (B, OC, H + 2 * pad[0] - KH + 1, W + 2 * pad[1] - KW + 1))
    d64 = oracle.conv2d_backward_data64(dy, w, (B, IC, H, W), stride, pad)
    ref = oracle.conv2d_backward_data_ref(dy, w, (B, IC, H, W), stride, pad)
    say("conv direct backward data", g)
    dx = host(ops().conv2d_backward_data(dev(dy), dev(w), (B, IC, H, W), stride, pad))
    assert oracle.rel_fro(dx, d64) <= 2 * oracle.rel_fro(ref, d64) + F32_FLOOR


@pytest.mark.parametrize("B,IC,OC,H,W", [(1, 10, 96, 14, 14), (3, 53, 64, 6, 7), (2, 64, 128, 28, 28),
                                         (1, 128, 16, 1, 1), (5, 1, 3, 3, 3), (2, 40, 1, 9, 9)])
@pytest.mark.parametrize("prec", [0, 1])
def test_1x1_is_a_product(B, IC, OC, H, W, prec):
    """Forward with and without bias and backward data of unpadded stride-1 1x1 layers; the
    operands are read as they lie, with a caller workspace and without."""
    import torch
    rng = np.random.default_rng(B + IC + OC + H)
    x, w = normal(rng, (B, IC, H, W)), normal(rng, (OC, IC, 1, 1), IC ** -0.5)
    b, dy = normal(rng, (OC,)), normal(rng, (B, OC, H, W))
    say("conv 1x1", B, IC, OC, H, W, prec)
    for bias in (b, None):
        y64 = oracle.conv2d_direct64(x, w, bias, (1, 1), (0, 0))
        ref = oracle.conv2d_ref_implicit(x, w, bias, (1, 1), (0, 0))
        y = host(ops().conv2d_forward(dev(x), dev(w), None if bias is None else dev(bias), (1, 1),
                                      (0, 0), precision=prec))
        assert oracle.rel_fro(y, y64) <= 2 * oracle.rel_fro(ref, y64) + F32_FLOOR
    d64 = oracle.conv2d_backward_data64(dy, w, x.shape, (1, 1), (0, 0))
    ref = oracle.conv2d_backward_data_ref(dy, w, x.shape, (1, 1), (0, 0))
    n = ops().conv2d_backward_data_workspace_bytes(x.shape, w.shape)
    ws = torch.empty(n // 4, device="cuda")
    d = ops().conv2d_backward_data(dev(dy), dev(w), x.shape, precision=prec)
    assert oracle.rel_fro(host(d), d64) <= 2 * oracle.rel_fro(ref, d64) + F32_FLOOR
    assert torch.equal(d, ops().conv2d_backward_data(dev(dy), dev(w), x.shape, precision=prec,
                                                     workspace=ws))


def test_small_3x3_routing():
    """Auto takes the direct kernel for small 3x3 stride-1 layers (forward in every mode, backward
    data in the TF32 modes), Winograd for the rest."""
    from cudeep_amd import cuDeep as cd
    from cudeep_amd.cuDeep import _core
    rng = np.random.default_rng(3)
    x, w = normal(rng, (2, 16, 12, 12)), normal(rng, (24, 16, 3, 3), 0.1)
    g = normal(rng, (2, 24, 12, 12))
    X, W, G = (_core.Tensor.from_numpy(a) for a in (x, w, g))
    prev, prec = cd.get_conv_algorithm(), cd.get_matmul_precision()
    say("small 3x3 routing")
    try:
        cd.set_matmul_precision("tf32")
        cd.set_conv_algorithm("auto")
        y = _core.conv2d_forward(X, W, None, [1, 1], [1, 1]).numpy()
        d = _core.conv2d_backward_data(G, W, [2, 16, 12, 12], [1, 1], [1, 1]).numpy()
        cd.set_conv_algorithm("implicit")
        assert np.array_equal(y, _core.conv2d_forward(X, W, None, [1, 1], [1, 1]).numpy())
        assert np.array_equal(d, _core.conv2d_backward_data(G, W, [2, 16, 12, 12], [1, 1],
                                                            [1, 1]).numpy())
    finally:
        cd.set_conv_algorithm(prev)
        cd.set_matmul_precision(prec)
    y64 = oracle.conv2d_direct64(x, w, None, (1, 1), (1, 1))
    assert oracle.rel_fro(y, y64) <= 2 * oracle.rel_fro(
        oracle.conv2d_ref_implicit(x, w, None, (1, 1), (1, 1)), y64)
