"""The FP32 GEMM at the sizes of the three-part kernel (gemm_parts.hip): the edges of its tiles and
k-tiles, its k-slices, the ones column, and operands outside the range in which its parts are
exact (recomputed on the fp32 matrix path).  Where k is short the product may run on another
kernel; test_gpu_gemm_parts_edges.py holds sizes that do not.  Bar throughout: relative Frobenius error against
fp64 within twice that of the reference's sequential fp32 FMA chain on the same operands (plus
one rounding where K < 64, as for the other FP32 kernels)."""
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


def _check(C, A, B, tA, tB, rows):
    """`rows` of C against fp64, at the bar above."""
    opA = np.ascontiguousarray((A.T if tA else A)[rows])
    C64 = oracle.dgemm(opA, B, False, tB)
    e_ref = oracle.rel_fro(oracle.sgemm_seqfma(opA, B, False, tB), C64)
    e = oracle.rel_fro(np.ascontiguousarray(C[rows]), C64)
    assert e <= 2 * e_ref + (F32_FLOOR if opA.shape[1] < 64 else 0.0), (e, e_ref)


def _rows(M):
    return sorted(set(range(0, 24)) | set(range(min(M, 120), min(M, 136))) | set(range(M - 24, M)))


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 32), (1921, 2050, 33), (2047, 2049, 17),
                                   (1926, 1925, 100), (2050, 2047, 31), (2048, 2176, 63)])
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
def test_edges(M, N, K, tA, tB):
    """Tiles that end 1-3 short of, at and past the edge; k-tails of 1, 4, 17 and 31; rows that
    start at any 4-byte alignment."""
    rng = np.random.default_rng(M + N + K)
    A = normal(rng, (K, M) if tA else (M, K))
    B = normal(rng, (N, K) if tB else (K, N))
    say("gemm parts", M, N, K, tA, tB)
    C = host(ops().gemm(dev(A), dev(B), transA=tA, transB=tB))
    assert np.isfinite(C).all()
    _check(C, A, B, tA, tB, _rows(M))
    # every column of every row: the row sums, each a sum of N outputs
    s64 = (A.T if tA else A).astype(np.float64) @ (B.T if tB else B).astype(np.float64).sum(1)
    assert oracle.rel_fro(C.astype(np.float64).sum(1), s64) < 1e-5


def test_views_and_epilogues():
    """Operands, output and aux with their own leading dimensions, nothing written outside the
    output; a fused bias + ReLU and a ReLU-backward epilogue equal the separate operations."""
    import torch
    import cudeep_amd as cd
    M, N, K = 2049, 2045, 70
    rng = np.random.default_rng(5)
    A = dev(normal(rng, (M, K + 3)))[:, 1:K + 1]
    B = dev(normal(rng, (K, N + 5)))[:, 2:N + 2]
    buf = torch.full((M + 2, N + 7), -7.0, device="cuda")
    say("gemm parts views")
    out = ops().gemm(A, B, out=buf[1:M + 1, 3:N + 3])
    plain = ops().gemm(A.contiguous(), B.contiguous())
    assert torch.equal(out, plain)
    inside = torch.zeros_like(buf, dtype=torch.bool)
    inside[1:M + 1, 3:N + 3] = True
    assert bool((buf[~inside] == -7.0).all())
    _check(host(plain), host(A.contiguous()), host(B.contiguous()), False, False, _rows(M))
    bias, aux = dev(normal(rng, (N,))), dev(normal(rng, (M, N + 1)))[:, :N]
    fused = ops().gemm(A, B, bias=bias, bias_mode=cd.BIAS_COL, epilogue=cd.EPI_RELU)
    assert torch.equal(fused, (plain + bias).relu())
    masked = ops().gemm(A, B, epilogue=cd.EPI_BWD_RELU, aux=aux)
    assert torch.equal(masked, torch.where(aux > 0, plain, torch.zeros_like(plain)))


@pytest.mark.parametrize("M,N,K", [(256, 784, 8192), (130, 256, 2049), (257, 255, 4099)])
@pytest.mark.parametrize("tB", [False, True])
def test_slices_with_ones_column(M, N, K, tB):
    """k-slices (the last one ragged) and the ones column inside, at the end of and past the
    tiles of op(B)'s own columns; the product itself is the same bits without it."""
    import torch
    rng = np.random.default_rng(M + K)
    A, B = normal(rng, (K, M)), normal(rng, (N, K) if tB else (K, N))
    cs = torch.full((M,), float("nan"), device="cuda")
    say("gemm parts slices", M, N, K, tB)
    C = ops().gemm(dev(A), dev(B), transA=True, transB=tB, colsum=cs)
    assert torch.equal(C, ops().gemm(dev(A), dev(B), transA=True, transB=tB))
    _check(host(C), A, B, True, tB, list(range(M)))
    db64 = A.astype(np.float64).sum(0)
    assert oracle.rel_fro(host(cs), db64) <= 2 * oracle.rel_fro(oracle.colsum(A), db64) + 2.0 ** -24


@pytest.mark.parametrize("M,N,K", [(1000, 1001, 4097), (1029, 1150, 2331)])
def test_slices_and_workspaces(M, N, K):
    """Own slices with ragged tiles and k, on a workspace of the queried size and on one too small
    for them (the product then takes another route, with as good a result)."""
    import torch
    rng = np.random.default_rng(M + K)
    A, B = normal(rng, (M, K)), normal(rng, (N, K))
    need = ops().gemm_workspace_bytes(M, N, K, transB=True)
    say("gemm parts workspaces", M, N, K, need)
    C = ops().gemm(dev(A), dev(B), transB=True)
    _check(host(C), A, B, False, True, _rows(M))
    assert need > 0
    ws = torch.empty(need // 4, device="cuda")
    assert torch.equal(C, ops().gemm(dev(A), dev(B), transB=True, workspace=ws))
    _check(host(ops().gemm(dev(A), dev(B), transB=True, workspace=ws[:4])), A, B, False, True,
           _rows(M))


@pytest.mark.parametrize("sa,sb", [(-118, 20), (-118, 100), (60, -70), (20, -118), (-60, -50),
                                   (-135, 30), (35, -140)])
def test_scales(sa, sb):
    """Operands scaled by powers of two, out of the range of exact parts on one side or both
    (and products near the smallest normal number, subnormal operands): the same bar."""
    M, N, K = 2048, 2048, 96
    rng = np.random.default_rng(77)
    A = (normal(rng, (M, K)) * np.float32(2.0) ** sa).astype(np.float32)
    B = (normal(rng, (K, N)) * np.float32(2.0) ** sb).astype(np.float32)
    say("gemm parts scales", sa, sb)
    C = host(ops().gemm(dev(A), dev(B)))
    _check(C, A, B, False, False, _rows(M))


def test_zero_outputs():
    """Zero rows and columns stay zero; a row of subnormals among them is not taken for one."""
    M, N, K = 2048, 2050, 70
    rng = np.random.default_rng(79)
    A, B = normal(rng, (M, K)), normal(rng, (K, N)) * np.float32(2.0 ** 20)
    A[3], A[130], B[:, 2049] = 0.0, 0.0, 0.0
    A[7] = (normal(rng, (K,)).astype(np.float64) * 2.0 ** -139).astype(np.float32)
    say("gemm parts zero outputs")
    C = host(ops().gemm(dev(A), dev(B)))
    assert not C[3].any() and not C[130].any() and not C[:, 2049].any()
    for r in (2, 7, 131):
        _check(C, A, B, False, False, [r])


def test_mixed_rows():
    """Rows and columns of very different size in one tile: every row to its own bar."""
    M, N, K = 2048, 2048, 128
    rng = np.random.default_rng(78)
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    A[5] *= np.float32(2.0 ** -115)
    A[140] *= np.float32(2.0 ** -122)
    A[300] = 0.0
    A[500, 3] = 3.4028234e38
    B[:, 700] *= np.float32(2.0 ** -117)
    say("gemm parts mixed rows")
    C = host(ops().gemm(dev(A), dev(B)))
    for r in (0, 5, 140, 299, 500):
        _check(C, A, B, False, False, [r])
    assert not C[300].any()
    col = np.ascontiguousarray(B[:, 700:701])
    C64 = oracle.dgemm(A[:64], col)
    e_ref = oracle.rel_fro(oracle.sgemm_seqfma(A[:64], col), C64)
    assert oracle.rel_fro(C[:64, 700:701], C64) <= 2 * e_ref
    # infinities and NaN: IEEE
    A[7, 2], A[9, 4] = np.inf, np.nan
    C = host(ops().gemm(dev(A), dev(B)))
    with np.errstate(invalid="ignore", over="ignore"):
        C64 = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(C), np.isnan(C64))
    big = np.abs(C64) > 3.4028234e38
    assert np.array_equal(np.isinf(C[~big]), np.isinf(C64[~big]))
    assert np.array_equal(np.sign(C[7]), np.sign(C64[7]))
