"""The convolution kernels that tile larger layers, at ragged sizes that their rules keep for them
(each test asserts the kernel): the row-window kernel (masked channel chunks, lanes of consecutive
pixels, strides, two-level sums in backward data), the gathering forward, the row-staged and the
gathering weight gradient.  Bar: error against fp64 within twice that of the reference's own route
(plus one rounding)."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import dev, host, normal, require_gpu, say
from tests.routes import conv_kernel

pytestmark = pytest.mark.gpu

FLOOR = 2.0 ** -24


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def ops():
    import cudeep_amd.ops as o
    return o


def _operands(g, seed):
    B, IC, OC, H, W, KH, KW, stride, pad = g
    rng = np.random.default_rng(seed + sum(g[:7]))
    oh, ow = (H + 2 * pad[0] - KH) // stride[0] + 1, (W + 2 * pad[1] - KW) // stride[1] + 1
    return (normal(rng, (B, IC, H, W)), normal(rng, (OC, IC, KH, KW), (2.0 / (IC * KH * KW)) ** 0.5),
            normal(rng, (OC,), 0.1), normal(rng, (B, OC, oh, ow)))


# batch, IC, OC, H, W, KH, KW, stride, padding
FORWARD = [
    ((46, 17, 65, 9, 40, 3, 3, (1, 1), (1, 1)), "rowwin"),     # 8 and 5 divide 40; masked chunk
    ((12, 24, 130, 13, 56, 3, 3, (1, 1), (1, 1)), "rowwin"),   # 8 and 7; tiles run past the image
    ((24, 3, 100, 11, 35, 3, 3, (1, 1), (1, 1)), "rowwin"),    # 7 and 5; k = 27
    ((20, 24, 100, 7, 70, 5, 5, (1, 1), (2, 2)), "rowwin"),
    ((27, 40, 64, 6, 120, 3, 3, (1, 1), (1, 1)), "rowwin"),    # wider window
    ((24, 8, 80, 10, 56, 3, 3, (1, 1), (0, 1)), "rowwin"),
    ((31, 5, 96, 23, 31, 5, 3, (2, 1), (2, 0)), "rowwin"),     # stride in one direction
    ((40, 20, 72, 30, 34, 3, 3, (2, 2), (1, 1)), "rowwin"),
    ((40, 9, 180, 14, 14, 7, 7, (1, 1), (3, 3)), "rowwin"),
    ((10, 40, 72, 12, 100, 5, 5, (1, 1), (2, 2)), "rowwin"),   # 5 chunks of 8 channels, wide window
    ((48, 8, 24, 20, 32, 3, 3, (1, 1), (1, 1)), "rowwin"),     # 128-pixel tiles
    ((42, 8, 24, 20, 32, 3, 3, (1, 1), (1, 1)), "rowwin"),     # 112
    ((2, 3, 20, 7, 1500, 3, 3, (1, 1), (1, 1)), "gather"),     # rows too wide for a window
    ((6, 15, 60, 7, 1600, 3, 3, (1, 1), (1, 1)), "gather"),
    ((2, 3, 40, 33, 1201, 5, 5, (2, 2), (2, 2)), "gather"),
]


@pytest.mark.parametrize("g,kernel", FORWARD)
def test_forward(g, kernel):
    assert conv_kernel("implicit", *g) == kernel
    x, w, b, _ = _operands(g, 0)
    stride, pad = g[7:]
    say("conv tiles forward", g, kernel)
    for bias in (b, None):
        y = host(ops().conv2d_implicit(dev(x), dev(w), None if bias is None else dev(bias), stride, pad))
        y64 = oracle.conv2d_direct64(x, w, bias, stride, pad)
        ref = oracle.conv2d_ref_implicit(x, w, bias, stride, pad)
        assert oracle.rel_fro(y, y64) <= 2 * oracle.rel_fro(ref, y64) + FLOOR


BACKWARD_DATA = [
    (26, 70, 24, 9, 40, 3, 3, (1, 1), (1, 1)),
    (12, 130, 33, 13, 56, 3, 3, (1, 1), (1, 1)),
    (26, 100, 17, 11, 35, 3, 3, (1, 1), (2, 0)),      # padding as wide as the filter allows
    (20, 90, 16, 9, 72, 5, 5, (1, 1), (2, 2)),
    (30, 65, 15, 9, 35, 5, 3, (1, 1), (4, 1)),
    (27, 64, 40, 6, 120, 3, 3, (1, 1), (1, 1)),
    (48, 72, 16, 10, 32, 3, 3, (1, 1), (1, 1)),
    (48, 24, 16, 20, 32, 3, 3, (1, 1), (1, 1)),
    (42, 24, 16, 20, 32, 3, 3, (1, 1), (1, 1)),
]


@pytest.mark.parametrize("g", BACKWARD_DATA)
@pytest.mark.parametrize("prec", [0, 1])
def test_backward_data(g, prec):
    assert conv_kernel("data", *g) == "rowwin"
    x, w, _, dy = _operands(g, 1)
    say("conv tiles backward data", g, prec)
    dx = host(ops().conv2d_backward_data(dev(dy), dev(w), x.shape, *g[7:], precision=prec))
    d64 = oracle.conv2d_backward_data64(dy, w, x.shape, *g[7:])
    ref = oracle.conv2d_backward_data_ref(dy, w, x.shape, *g[7:])
    assert oracle.rel_fro(dx, d64) <= 2 * oracle.rel_fro(ref, d64) + FLOOR


BACKWARD_WEIGHT = [
    ((10, 20, 70, 31, 30, 3, 3, (1, 1), (2, 2)), "rows"),      # ragged channels, pad 2, rows of 32
    ((12, 20, 100, 20, 70, 3, 3, (1, 1), (1, 1)), "rows"),     # two segments per row
    ((9, 16, 80, 30, 61, 3, 3, (1, 1), (1, 1)), "rows"),       # 61 of 64 pixels
    ((7, 33, 66, 40, 54, 3, 3, (1, 1), (0, 1)), "rows"),       # 56-pixel segments, no pad above
    ((60, 64, 70, 20, 29, 3, 3, (1, 1), (1, 0)), "rows"),      # 64-channel tile
    ((46, 21, 192, 25, 27, 3, 3, (2, 1), (1, 1)), "gather"),
    ((60, 13, 180, 19, 23, 5, 3, (1, 1), (2, 1)), "gather"),   # 195 filter elements, 180 channels
]


@pytest.mark.parametrize("g,kernel", BACKWARD_WEIGHT)
def test_backward_weight(g, kernel):
    import torch
    assert conv_kernel("weight", *g) == kernel
    x, w, _, dy = _operands(g, 2)
    say("conv tiles backward weight", g, kernel)
    dw = ops().conv2d_backward_weight(dev(dy), dev(x), w.shape, *g[7:])
    d64 = oracle.conv2d_backward_weight64(dy, x, w.shape, *g[7:])
    ref = oracle.conv2d_backward_weight_ref(dy, x, w.shape, *g[7:])
    assert oracle.rel_fro(host(dw), d64) <= 2 * oracle.rel_fro(ref, d64) + FLOOR
    n = ops().conv2d_backward_weight_workspace_bytes(x.shape, w.shape, *g[7:])
    ws = torch.full((n // 4 + 1,), float("nan"), device="cuda")
    assert torch.equal(dw, ops().conv2d_backward_weight(dev(dy), dev(x), w.shape, *g[7:], workspace=ws))
    from cudeep_amd import _lib as L   # and the entry point that never allocates
    B, IC, OC, H, W, KH, KW, stride, pad = g
    again, gx, gdy = torch.full_like(dw, float("nan")), dev(x), dev(dy)
    L.call("cdx_conv2d_backward_weight_f32_noalloc", gdy.data_ptr(), gx.data_ptr(), again.data_ptr(), B,
           IC, OC, H, W, KH, KW, *stride, *pad, 0, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(dw, again)
