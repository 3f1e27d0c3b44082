"""Split-precision and 16-bit GEMMs whose rows and columns are whole tiles and whose k is not: the
last, partial k-tile runs checked after the unchecked loop.  One, two, three and more k-tiles
before it (each ends the pipelined loop differently), tails of 1, 4 and all but one k."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import dev, host, normal, require_gpu, say

pytestmark = pytest.mark.gpu

# 2048 x 2048 runs 128 x 128 tiles, 768 x 768 64 x 64 ones, 64 x 4160 the 64 x 128 ones (k-tile 32)
SIZES = [(2048, 2048, 68), (2048, 2048, 196), (768, 768, 127), (768, 768, 129), (768, 832, 252),
         (768, 768, 324), (64, 4096, 36), (64, 4096, 127)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("kind", ["tf32", "tf32x4", "bf16"])
def test_k_tail(M, N, K, tA, tB, kind):
    require_gpu()
    import torch
    import cudeep_amd as cd
    import cudeep_amd.ops as ops
    rng = np.random.default_rng(M + N + K + 2 * tA + tB)
    ld = (K + 7) // 8 * 8   # 16-byte rows whatever K
    A = normal(rng, (K, M) if tA else (M, ld))
    B = normal(rng, (N, ld) if tB else (K, N))
    dA, dB = dev(A), dev(B)
    if kind == "bf16":
        dA, dB = dA.to(torch.bfloat16), dB.to(torch.bfloat16)
        A, B = host(dA.float()), host(dB.float())
    va, vb = (dA if tA else dA[:, :K]), (dB[:, :K] if tB else dB)
    # what lies behind the rows is not read into the sums
    if not tA and ld > K:
        dA[:, K:] = float("nan")
    if tB and ld > K:
        dB[:, K:] = float("nan")
    say("gemm k tail", M, N, K, tA, tB, kind)
    if kind == "bf16":
        C = host(ops.gemm16(va, vb, transA=tA, transB=tB))
    else:
        C = host(ops.gemm(va, vb, transA=tA, transB=tB,
                          precision=cd.PREC_TF32MODE if kind == "tf32" else cd.PREC_TF32MODE4))
    rows = sorted({0, 1, 63, 64 % M, M // 2 + 1, M - 1})
    opA = np.ascontiguousarray((A.T if tA else A[:, :K])[rows])
    opB = np.ascontiguousarray(B[:, :K].T if tB else B)
    C64 = oracle.dgemm(opA, opB)
    bar = min(oracle.rel_fro(oracle.gemm_tf32emu(opA, opB, m), C64) for m in ("rz", "rne"))
    # (16-bit operands: the emulation is the ideal MMA, to within twice)
    assert oracle.rel_fro(C[rows], C64) <= (2 * bar if kind == "bf16" else bar)
