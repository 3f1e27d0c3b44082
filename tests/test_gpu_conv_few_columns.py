"""Forward convolutions below 4 MiB of columns that keep the column route: a long k (the product in
slices), layers that only the tiling implicit kernels would take, more taps than the direct kernel's
mask.  FP32 products in every precision mode; with a caller workspace of the queried size, which
holds the slices too, of the columns alone, and without.  Captured on the queried workspace, replays
equal the eager call.  Against fp64 within twice the error of the reference's own route."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import F32_FLOOR, dev, host, normal, require_gpu, say
from tests.routes import conv_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", [(1, 161, 33, 14, 15, 5, 5, (2, 2), (2, 2)),
                               (2, 82, 48, 9, 9, 7, 7, (2, 2), (3, 3)),
                               (4, 65, 513, 56, 56, 1, 1, (2, 2), (0, 0)),
                               (1, 12, 40, 13, 13, 11, 11, (4, 4), (5, 5))])
@pytest.mark.parametrize("prec", [0, 1, 2])
def test_forward(g, prec):
    require_gpu()
    import torch
    import cudeep_amd.ops as ops
    from cudeep_amd import _lib as L
    assert conv_kernel("forward", *g) == "im2col"
    B, IC, OC, H, W, KH, KW, stride, pad = g
    rng = np.random.default_rng(sum(g[:7]))
    x, w = normal(rng, (B, IC, H, W)), normal(rng, (OC, IC, KH, KW), (2.0 / (IC * KH * KW)) ** 0.5)
    b = normal(rng, (OC,))
    say("conv few columns", g, prec)
    y = ops.conv2d_forward(dev(x), dev(w), dev(b), stride, pad, precision=prec)
    y64 = oracle.conv2d_direct64(x, w, b, stride, pad)
    ref = oracle.conv2d_ref_im2col(x, w, b, stride, pad)
    assert oracle.rel_fro(host(y), y64) <= 2 * oracle.rel_fro(ref, y64) + F32_FLOOR
    n = L.lib().cdx_conv2d_forward_workspace_size(B, IC, H, W, KH, KW, *stride, *pad)
    ws = torch.full((n // 4,), float("nan"), device="cuda")
    assert n > 0 and torch.equal(y, ops.conv2d_forward(dev(x), dev(w), dev(b), stride, pad,
                                                       precision=prec, workspace=ws))
    S = y64.shape[2] * y64.shape[3]
    cols = ws[:IC * KH * KW * B * S]
    assert torch.equal(y, ops.conv2d_forward(dev(x), dev(w), dev(b), stride, pad, precision=prec,
                                             workspace=cols))


@pytest.mark.parametrize("g", [(1, 161, 33, 14, 15, 5, 5, (2, 2), (2, 2)),
                               (1, 24, 40, 13, 13, 11, 11, (4, 4), (5, 5)),
                               (1, 20, 640, 13, 13, 11, 11, (4, 4), (5, 5))])
def test_capture(g):
    require_gpu()
    import torch
    import cudeep_amd.ops as ops
    from cudeep_amd import _lib as L
    B, IC, OC, H, W, KH, KW, stride, pad = g
    rng = np.random.default_rng(sum(g[:7]))
    x, w = dev(normal(rng, (B, IC, H, W))), dev(normal(rng, (OC, IC, KH, KW)))
    n = L.lib().cdx_conv2d_forward_workspace_size(B, IC, H, W, KH, KW, *stride, *pad)
    ws = torch.empty(n // 4, device="cuda")
    say("conv few columns capture", g)
    out = ops.conv2d_forward(x, w, None, stride, pad, workspace=ws)

    def step():
        ops.conv2d_forward(x, w, None, stride, pad, workspace=ws, out=out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for r in range(3):
        x.mul_(-2.0)
        out.fill_(float("nan"))
        say("conv few columns replay", r)
        graph.replay()
        torch.cuda.synchronize()
        y = out.clone()
        step()
        torch.cuda.synchronize()
        assert torch.equal(y, out)
