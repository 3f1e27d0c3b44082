"""The FP32 GEMM on three exact bf16 parts per operand (gemm_parts.hip) at sizes that its rule keeps
for it: tile and k-tile edges, views and epilogues, batches, the ones column.  Each test asserts
the kernel.  Bar: relative Frobenius error against fp64 within twice that of the reference's
sequential fp32 FMA chain on the same operands."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import dev, host, normal, require_gpu, say
from tests.routes import gemm_kernel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def ops():
    import cudeep_amd.ops as o
    return o


def _rows(M):
    return sorted(set(range(0, 12)) | set(range(min(M, 122), min(M, 134))) | set(range(M - 12, M)))


def _check(C, A, B, tA, tB, rows):
    opA = np.ascontiguousarray((A.T if tA else A)[rows])
    C64 = oracle.dgemm(opA, B, False, tB)
    e_ref = oracle.rel_fro(oracle.sgemm_seqfma(opA, B, False, tB), C64)
    assert oracle.rel_fro(np.ascontiguousarray(C[rows]), C64) <= 2 * e_ref


# k-tiles of 32: tails of 1, 4, 17, 31 and none, odd and even counts; rows and columns 1 to 3 short
# of, at and past a 128-tile
@pytest.mark.parametrize("M,N,K", [(2048, 2048, 96), (2047, 1921, 97), (1921, 2047, 132),
                                   (1926, 1925, 324), (2047, 2049, 337), (2050, 2047, 351),
                                   (1921, 2050, 641)])
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
def test_edges(M, N, K, tA, tB):
    assert gemm_kernel(0, M, N, K, tA, tB) == "parts"
    rng = np.random.default_rng(M + N + K)
    A = normal(rng, (K, M) if tA else (M, K))
    B = normal(rng, (N, K) if tB else (K, N))
    say("gemm parts edges", M, N, K, tA, tB)
    C = host(ops().gemm(dev(A), dev(B), transA=tA, transB=tB))
    assert np.isfinite(C).all()
    _check(C, A, B, tA, tB, _rows(M))
    # every column of every row: the row sums, each a sum of N outputs
    s64 = (A.T if tA else A).astype(np.float64) @ (B.T if tB else B).astype(np.float64).sum(1)
    assert oracle.rel_fro(C.astype(np.float64).sum(1), s64) < 1e-5


def test_views_and_epilogues():
    """Operands, output and aux with their own leading dimensions; nothing written outside."""
    import torch
    import cudeep_amd as cd
    M, N, K = 2049, 2045, 390
    assert gemm_kernel(0, M, N, K, lda=K + 3, ldb=N + 5) == "parts"
    rng = np.random.default_rng(5)
    A = dev(normal(rng, (M, K + 3)))[:, 1:K + 1]
    B = dev(normal(rng, (K, N + 5)))[:, 2:N + 2]
    buf = torch.full((M + 2, N + 7), -7.0, device="cuda")
    say("gemm parts views at K = 390")
    out = ops().gemm(A, B, out=buf[1:M + 1, 3:N + 3])
    plain = ops().gemm(A.contiguous(), B.contiguous())
    assert torch.equal(out, plain)
    inside = torch.zeros_like(buf, dtype=torch.bool)
    inside[1:M + 1, 3:N + 3] = True
    assert bool((buf[~inside] == -7.0).all())
    bias, aux = dev(normal(rng, (N,))), dev(normal(rng, (M, N + 1)))[:, :N]
    fused = ops().gemm(A, B, bias=bias, bias_mode=cd.BIAS_COL, epilogue=cd.EPI_RELU)
    assert torch.equal(fused, (plain + bias).relu())
    masked = ops().gemm(A, B, epilogue=cd.EPI_BWD_RELU, aux=aux)
    assert torch.equal(masked, torch.where(aux > 0, plain, torch.zeros_like(plain)))


def test_batch():
    """Three products in one launch (a 1x1 convolution of 320 -> 512 channels on 97 x 101
    pixels): each image to its own bar, rows that start at any 4-byte alignment."""
    import torch
    B, IC, OC, H, W = 3, 320, 512, 97, 101
    rng = np.random.default_rng(11)
    x, w = dev(normal(rng, (B, IC, H, W))), dev(normal(rng, (OC, IC, 1, 1), IC ** -0.5))
    bias = dev(normal(rng, (OC,)))
    say("gemm parts batch")
    y = ops().conv2d_forward(x, w, bias, (1, 1), (0, 0)).view(B, OC, H * W)
    for b in range(B):
        want = w.view(OC, IC).double() @ x[b].view(IC, H * W).double() + bias.double()[:, None]
        one = torch.matmul(w.view(OC, IC).cpu(), x[b].view(IC, H * W)[:, ::97].contiguous().cpu()) \
            + bias.cpu()[:, None]
        ref = want[:, ::97].cpu()
        e_ref = float((one.double() - ref).norm() / ref.norm())
        assert float((y[b].double() - want).norm() / want.norm()) <= 2 * e_ref
