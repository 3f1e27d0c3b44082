"""1x1 layers of one image whose product would run in k-slices, in scratch of its own: they take a
kernel that needs none, so that a call with the workspace that was asked for allocates nothing and
can be captured.  Against fp64 within twice the error of the reference's route; replays of a
captured forward and backward data pass equal the eager calls bit for bit."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import dev, host, normal, require_gpu, say
from tests.routes import conv_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("IC,OC,H,W", [(2048, 64, 28, 28), (64, 2050, 20, 19), (1030, 16, 13, 9),
                                       (2100, 2048, 7, 7)])
def test_one_image_long_k(IC, OC, H, W):
    require_gpu()
    import torch
    import cudeep_amd.ops as ops
    from cudeep_amd import _lib as L
    g = (1, IC, OC, H, W, 1, 1)
    if IC >= 1024:
        assert conv_kernel("forward", *g) == "direct"
    if OC >= 1024:
        assert conv_kernel("data", *g) == "direct"
    rng = np.random.default_rng(IC + OC)
    x, w = normal(rng, (1, IC, H, W)), normal(rng, (OC, IC, 1, 1), IC ** -0.5)
    b, dy = normal(rng, (OC,)), normal(rng, (1, OC, H, W))
    dx_, dw_, db_, dyd = dev(x), dev(w), dev(b), dev(dy)
    n = L.lib().cdx_conv2d_forward_workspace_size(1, IC, H, W, 1, 1, 1, 1, 0, 0)
    ws = torch.empty(n // 4 + 1, device="cuda")
    wd = torch.empty(ops.conv2d_backward_data_workspace_bytes(x.shape, w.shape) // 4, device="cuda")
    out, grad = torch.empty((1, OC, H, W), device="cuda"), torch.empty((1, IC, H, W), device="cuda")

    def step():
        ops.conv2d_forward(dx_, dw_, db_, (1, 1), (0, 0), workspace=ws, out=out)
        ops.conv2d_backward_data(dyd, dw_, x.shape, workspace=wd, out=grad)
    say("conv 1x1 long k", IC, OC, H, W)
    step()
    y, d = out.clone(), grad.clone()
    y64 = oracle.conv2d_direct64(x, w, b, (1, 1), (0, 0))
    ref = oracle.conv2d_ref_implicit(x, w, b, (1, 1), (0, 0))
    assert oracle.rel_fro(host(y), y64) <= 2 * oracle.rel_fro(ref, y64)
    d64 = oracle.conv2d_backward_data64(dy, w, x.shape, (1, 1), (0, 0))
    ref = oracle.conv2d_backward_data_ref(dy, w, x.shape, (1, 1), (0, 0))
    assert oracle.rel_fro(host(d), d64) <= 2 * oracle.rel_fro(ref, d64)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for r in range(3):
        dx_.mul_(-1.0)
        dyd.mul_(2.0)
        out.fill_(float("nan"))
        grad.fill_(float("nan"))
        say("conv 1x1 long k replay", r)
        graph.replay()
        torch.cuda.synchronize()
        y, d = out.clone(), grad.clone()
        step()
        torch.cuda.synchronize()
        assert torch.equal(y, out) and torch.equal(d, grad)
