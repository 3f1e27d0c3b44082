"""The split-precision (TF32-mode) and tiled 16-bit kernels at ragged sizes beyond those that the
unstaged kernels take (each test asserts the kernel): checked loads, rows at any 4-byte alignment,
edges, bias and activation, nothing written outside, and the repair of outputs that an infinite or
out-of-range operand reaches.  Bar: error against fp64 within that of the reference's TF32
(16-bit: twice that of the ideal product of the same operands)."""
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
    return sorted({r for r in (0, 1, 63, 64, 127, 128, M // 2, M - 65, M - 2, M - 1) if 0 <= r < M})


# unaligned rows or k: more than 1024 tiles of 32 x 32; aligned ones: more than 256
@pytest.mark.parametrize("M,N,K", [(1023, 1300, 333), (1100, 1051, 65), (700, 900, 300), (66, 12001, 201),
                                   (2050, 2047, 127)])
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("prec", [1, 2])
def test_tf32(M, N, K, tA, tB, prec):
    import torch
    import cudeep_amd as cd
    rng = np.random.default_rng(M + N + K + 2 * tA + tB)
    A = normal(rng, (K, M) if tA else (M, K))
    B = normal(rng, (N, K) if tB else (K, N))
    assert gemm_kernel(prec, M, N, K, tA, tB) == "split"
    say("gemm split ragged", M, N, K, tA, tB, prec)
    buf = torch.full((M + 2, N + 3), -7.0, device="cuda")
    C = ops().gemm(dev(A), dev(B), transA=tA, transB=tB, precision=prec, out=buf[1:M + 1, 2:N + 2])
    inside = torch.zeros_like(buf, dtype=torch.bool)
    inside[1:M + 1, 2:N + 2] = True
    assert bool((buf[~inside] == -7.0).all())
    rows = _rows(M)
    opA, opB = np.ascontiguousarray((A.T if tA else A)[rows]), np.ascontiguousarray(B.T if tB else B)
    C64 = oracle.dgemm(opA, opB)
    bar = min(oracle.rel_fro(oracle.gemm_tf32emu(opA, opB, m), C64) for m in ("rz", "rne"))
    assert oracle.rel_fro(host(C)[rows], C64) <= bar
    bias = dev(normal(rng, (N,)))
    fused = ops().gemm(dev(A), dev(B), transA=tA, transB=tB, precision=prec, bias=bias,
                       bias_mode=cd.BIAS_COL, epilogue=cd.EPI_RELU)
    assert torch.equal(fused, (C + bias).relu())


@pytest.mark.parametrize("prec", [1, 2])
def test_tf32_special_values(prec):
    """Infinities, NaN and the largest values: every output IEEE, as many as there are."""
    M, N, K = 1023, 1301, 333
    assert gemm_kernel(prec, M, N, K) == "split"
    rng = np.random.default_rng(prec)
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    A[3, 332], A[700, 1], A[900, 300], A[1022, 5] = np.inf, -np.inf, np.nan, 3.4e38
    B[5, 77], B[332, 9] = 0.5, 0.0
    say("gemm split special values", prec)
    C = host(ops().gemm(dev(A), dev(B), precision=prec))
    with np.errstate(invalid="ignore", over="ignore"):
        C64 = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(C), np.isnan(C64))
    assert np.array_equal(np.sign(C[3][~np.isnan(C[3])]), np.sign(C64[3][~np.isnan(C[3])]))
    assert np.isinf(C[3][~np.isnan(C[3])]).all() and np.isfinite(C[4]).all()


@pytest.mark.parametrize("M,N,K", [(900, 930, 131), (1601, 700, 65), (833, 4101, 40)])
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("bf16", [False, True])
def test_16bit(M, N, K, tA, tB, bf16):
    import torch
    dt = torch.bfloat16 if bf16 else torch.float16
    assert gemm_kernel("bf16" if bf16 else "f16", M, N, K, tA, tB) == "tiled"
    rng = np.random.default_rng(M + N + K + 2 * tA + tB)
    a = dev(normal(rng, (K, M) if tA else (M, K))).to(dt)
    b = dev(normal(rng, (N, K) if tB else (K, N), 0.2)).to(dt)
    say("gemm16 ragged", M, N, K, tA, tB, bf16)
    C = host(ops().gemm16(a, b, transA=tA, transB=tB))
    A, B = host(a.float()), host(b.float())
    rows = _rows(M)
    opA, opB = np.ascontiguousarray((A.T if tA else A)[rows]), np.ascontiguousarray(B.T if tB else B)
    C64 = oracle.dgemm(opA, opB)
    assert oracle.rel_fro(C[rows], C64) <= 2 * oracle.rel_fro(oracle.gemm_tf32emu(opA, opB, "rne"), C64)
