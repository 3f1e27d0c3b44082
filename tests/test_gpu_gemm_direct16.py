"""The 16-bit GEMM that reads its operands straight from global memory (gemm_direct16.hip): edges of
its 16- and 32-wide tiles, 32-k steps and k runs, leading dimensions that are even, multiples of 8
and odd (which keep the tiled route), epilogues.  Bar: relative Frobenius error against fp64 within
twice that of the ideal MMA on the same operands (the emulation forms their products exactly)."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import F32_FLOOR, dev, host, normal, require_gpu, say

pytestmark = pytest.mark.gpu

SIZES = [(1, 15, 8), (17, 16, 31), (16, 33, 32), (33, 31, 65), (70, 50, 127), (100, 100, 640),
         (63, 301, 417), (450, 300, 96), (510, 600, 130)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("bf16", [False, True])
def test_edges(M, N, K, tA, tB, bf16):
    require_gpu()
    import torch
    import cudeep_amd as cd
    import cudeep_amd.ops as ops
    dt = torch.bfloat16 if bf16 else torch.float16
    rng = np.random.default_rng(M + 3 * N + 7 * K + 2 * tA + tB)
    a = dev(normal(rng, (K, M) if tA else (M, K))).to(dt)
    b = dev(normal(rng, (N, K) if tB else (K, N), 0.2)).to(dt)
    A32, B32 = host(a.float()), host(b.float())
    opA, opB = np.ascontiguousarray(A32.T if tA else A32), np.ascontiguousarray(B32.T if tB else B32)
    C64 = oracle.dgemm(opA, opB)
    bar = 2 * oracle.rel_fro(oracle.gemm_tf32emu(opA, opB, "rne"), C64) + F32_FLOOR
    bias = dev(normal(rng, (N,)))
    for pad in (0, 1, 8):   # leading dimension past the row: any, odd or even, and 16-byte rows
        wa = torch.zeros((a.shape[0], a.shape[1] + pad), device="cuda", dtype=dt)
        wb = torch.zeros((b.shape[0], b.shape[1] + pad), device="cuda", dtype=dt)
        va, vb = wa[:, :a.shape[1]], wb[:, :b.shape[1]]
        va.copy_(a)
        vb.copy_(b)
        buf = torch.full((M + 2, N + 3), -7.0, device="cuda")
        say("gemm direct16", M, N, K, tA, tB, bf16, pad)
        C = ops.gemm16(va, vb, transA=tA, transB=tB, out=buf[1:M + 1, 2:N + 2])
        assert oracle.rel_fro(host(C), C64) <= bar
        fused = ops.gemm16(va, vb, transA=tA, transB=tB, bias=bias, bias_mode=cd.BIAS_COL,
                           epilogue=cd.EPI_RELU)
        assert torch.equal(fused, (C + bias).relu())
        inside = torch.zeros_like(buf, dtype=torch.bool)
        inside[1:M + 1, 2:N + 2] = True
        assert bool((buf[~inside] == -7.0).all())


def test_special_values():
    """Infinities and NaN before and in the last, partial step reach exactly their row."""
    require_gpu()
    import torch
    import cudeep_amd.ops as ops
    rng = np.random.default_rng(4)
    a = dev(normal(rng, (40, 75))).to(torch.bfloat16)
    b = dev(normal(rng, (75, 30))).to(torch.bfloat16)
    a[3, 74], a[5, 2], a[9, 70] = float("inf"), float("-inf"), float("nan")
    say("gemm direct16 special values")
    C = host(ops.gemm16(a, b))
    with np.errstate(invalid="ignore"):
        C64 = host(a.float()).astype(np.float64) @ host(b.float()).astype(np.float64)
    assert np.array_equal(np.isnan(C), np.isnan(C64))
    assert np.array_equal(np.isinf(C), np.isinf(C64))
    assert np.array_equal(np.sign(C[[3, 5]]), np.sign(C64[[3, 5]]))
