"""The FP32 GEMM that reads its operands straight from global memory (gemm_direct.hip): edges of
its 16- and 32-wide tiles, of its 16-k steps and of the four k runs of a split, any alignment,
batches of its calls' epilogues, and the ones column.  Bar: relative Frobenius error against fp64
within twice that of the reference's sequential fp32 FMA chain (plus one rounding where K < 64)."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import F32_FLOOR, dev, host, normal, require_gpu, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def ops():
    import cudeep_amd.ops as o
    return o


def _bar(A, B, tA, tB):
    C64 = oracle.dgemm(A, B, tA, tB)
    return C64, 2 * oracle.rel_fro(oracle.sgemm_seqfma(A, B, tA, tB), C64) + \
        (F32_FLOOR if (A.shape[0] if tA else A.shape[1]) < 64 else 0.0)


# (17 .. 127 k: no split; 128 and more: runs of 2, 2, 2, 2 steps, of 3, 3, 3, 1 with a tail, ...;
# up to 512 16 x 16 tiles and beyond)
SIZES = [(1, 17, 17), (17, 18, 31), (33, 31, 64), (15, 300, 127), (63, 65, 128), (100, 70, 161),
         (65, 33, 1533), (300, 200, 784), (511, 513, 130), (640, 609, 147), (765, 700, 37)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("pad", [0, 1, 3])
def test_edges(M, N, K, tA, tB, pad):
    """Operands at any 4-byte alignment and leading dimension, in both precision modes (exact
    products are inside the TF32 mode's bar too); nothing written outside the output."""
    import torch
    import cudeep_amd as cd
    rng = np.random.default_rng(M * 31 + N * 7 + K + pad)
    A = normal(rng, (K, M + pad) if tA else (M, K + pad))[:, pad:]
    B = normal(rng, (N, K + pad) if tB else (K, N + pad))[:, :(K if tB else N)]
    dA = torch.zeros((A.shape[0], A.shape[1] + pad), device="cuda")
    dB = torch.zeros((B.shape[0], B.shape[1] + 2 * pad), device="cuda")
    vA, vB = dA[:, pad:], dB[:, pad:pad + B.shape[1]]
    vA.copy_(dev(A))
    vB.copy_(dev(B))
    buf = torch.full((M + 2, N + 3), -7.0, device="cuda")
    out = buf[1:M + 1, 2:N + 2]
    say("gemm direct", M, N, K, tA, tB, pad)
    C = host(ops().gemm(vA, vB, transA=tA, transB=tB, out=out))
    C64, bar = _bar(A, B, tA, tB)
    assert oracle.rel_fro(C, C64) <= bar
    full = host(buf)
    full[1:M + 1, 2:N + 2] = -7.0
    assert (full == -7.0).all()
    if M * N <= 256 * 1024 and K > 16:
        T = host(ops().gemm(vA, vB, transA=tA, transB=tB, precision=cd.PREC_TF32MODE))
        emu = min(oracle.rel_fro(oracle.gemm_tf32emu(A.T if tA else A, B.T if tB else B, m), C64)
                  for m in ("rz", "rne"))
        assert oracle.rel_fro(T, C64) <= emu


@pytest.mark.parametrize("M,N,K", [(40, 33, 100), (200, 300, 700), (640, 600, 333)])
@pytest.mark.parametrize("tB", [False, True])
def test_epilogues_and_ones_column(M, N, K, tB):
    """Bias + activation and activation-backward epilogues equal the separate operations on the
    same product, bit for bit; so does the product beside the ones column, whose sums are within
    twice the serial fp32 column sum's error."""
    import torch
    import cudeep_amd as cd
    rng = np.random.default_rng(M + N + K)
    A, B = normal(rng, (K, M)), normal(rng, (N, K) if tB else (K, N))
    dA, dB = dev(A), dev(B)
    say("gemm direct epilogues", M, N, K, tB)
    plain = ops().gemm(dA, dB, transA=True, transB=tB)
    bias, aux = dev(normal(rng, (M,))), dev(normal(rng, (M, N)))
    fused = ops().gemm(dA, dB, transA=True, transB=tB, bias=bias, bias_mode=cd.BIAS_ROW,
                       epilogue=cd.EPI_RELU)
    assert torch.equal(fused, (plain + bias[:, None]).relu())
    masked = ops().gemm(dA, dB, transA=True, transB=tB, epilogue=cd.EPI_BWD_RELU, aux=aux)
    assert torch.equal(masked, torch.where(aux > 0, plain, torch.zeros_like(plain)))
    cs = torch.full((M,), float("nan"), device="cuda")
    assert torch.equal(ops().gemm(dA, dB, transA=True, transB=tB, colsum=cs), plain)
    db64 = A.astype(np.float64).sum(0)
    assert oracle.rel_fro(host(cs), db64) <= 2 * oracle.rel_fro(oracle.colsum(A), db64) + 2.0 ** -24


def test_special_values():
    """Infinities, NaN, the largest and subnormal operands in the last, partial step and before."""
    M, N, K = 70, 50, 203
    rng = np.random.default_rng(9)
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    A[3, 202], A[7, 1], A[9, 200] = np.inf, -np.inf, np.nan
    A[20, 5], A[21, 201] = 3.4e38, -3.4e38
    B[5], B[201] = 0.5, 0.25
    A[30] = 1e-42
    say("gemm direct special values")
    C = host(ops().gemm(dev(A), dev(B)))
    with np.errstate(invalid="ignore", over="ignore"):
        C64 = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(C), np.isnan(C64))
    assert np.array_equal(np.isinf(C), np.isinf(C64))
    assert np.array_equal(np.sign(C[3]), np.sign(C64[3]))
