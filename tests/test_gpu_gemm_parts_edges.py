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


# (the value, its row and column in A: 2^41 and a mask's -1e30 among N(0, 1), or a whole row)
@pytest.mark.parametrize("what", ["2^41", "-1e30", "1e-18 row", "1e30 in B", "zero and tiny rows"])
def test_outliers_leave_the_other_rows_alone(what):
    """One large value, or a row of small ones, does not send the tile's other outputs to the
    fp32 matrix path: they are the same bits as without it, and the row itself meets its bar."""
    import torch
    M, N, K = 2048, 2048, 160
    assert gemm_kernel(0, M, N, K) == "parts"
    rng = np.random.default_rng(21)
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    say("gemm parts outliers", what)
    base = ops().gemm(dev(A), dev(B))
    rows, cols = [5], []
    if what == "2^41":
        # (1.37: with a power of two the one large product is exact in the reference, whose error
        # is then not a rounding, 2^-24, but only what the rest of the sum is worth, 2^-37)
        A[5, 7] = 1.37 * 2.0 ** 41
    elif what == "-1e30":
        A[5, ::3] = -1e30
    elif what == "1e30 in B":
        B[7, 9] = 1e30
        rows, cols = [], [9]
    elif what == "1e-18 row":
        A[5] *= np.float32(1e-18)
    else:
        A[5] *= np.float32(1e-18)
        A[64:96] = 0.0
        rows = [5] + list(range(64, 96))
    C = ops().gemm(dev(A), dev(B))
    same = torch.ones((M, N), dtype=torch.bool, device="cuda")
    same[rows, :] = False
    same[:, cols] = False
    assert torch.equal(C[same], base[same])
    _check(host(C), A, B, False, False, [5])
    assert what != "zero and tiny rows" or not host(C)[64:96].any()


@pytest.mark.parametrize("sa,sb", [(-70, -44), (-109, -9), (-100, 2), (-60, -40), (100, -80),
                                   (-112, 60), (30, -111)])
def test_scales(sa, sb):
    """Operands scaled by powers of two on either side of the lines at which parts or their
    products would vanish, with values of other sizes beside them: every row to the bar."""
    M, N, K = 2048, 2048, 160
    rng = np.random.default_rng(22)
    A = (normal(rng, (M, K)).astype(np.float64) * 2.0 ** sa).astype(np.float32)
    B = (normal(rng, (K, N)).astype(np.float64) * 2.0 ** sb).astype(np.float32)
    A[9] *= np.float32(2.0 ** -12)
    A[140, 3] *= np.float32(2.0 ** 20)
    say("gemm parts scales", sa, sb)
    C = host(ops().gemm(dev(A), dev(B)))
    for rows in ([9], [140], list(range(16, 40))):
        _check(C, A, B, False, False, rows)


def test_infinite_and_overflowing_outputs():
    """Infinities, NaN, sums that overflow and values that bf16 would round to infinity: IEEE."""
    M, N, K = 2048, 2048, 160
    rng = np.random.default_rng(23)
    A, B = normal(rng, (M, K)), normal(rng, (K, N))
    A[3, 5], A[300, 9], A[600, 11] = np.inf, np.nan, 3.4028234e38
    A[900, :2], B[:2, 40] = 3e38, 1.0
    B[11] = 0.5
    say("gemm parts infinities")
    C = host(ops().gemm(dev(A), dev(B)))
    with np.errstate(invalid="ignore", over="ignore"):
        C64 = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(C), np.isnan(C64))
    assert np.array_equal(np.sign(C[3]), np.sign(C64[3])) and np.isinf(C[3]).all()
    assert np.isposinf(C[900, 40])
    _check(C, A, B, False, False, [600])


@pytest.mark.parametrize("tA,tB", [(False, False), (True, True)])
def test_one_product_per_output(tA, tB):
    """A diagonal, a permutation and powers of two.  An output that is one product ab misses the
    terms am bl + al bm + al bl, at most 2^-24 |ab|, and takes one rounding to one side, 2^-23, on
    the sum's way to 24 bits (the smaller terms' own roundings are 2^-8 of that); with one factor a
    power of two its m and l are 0 and nothing is lost."""
    M = N = K = 2048
    assert gemm_kernel(0, M, N, K, tA, tB) == "parts"
    rng = np.random.default_rng(31)
    B = normal(rng, (K, N))
    perm = rng.permutation(K)

    def product(A):
        return host(ops().gemm(dev(A.T if tA else A), dev(B.T if tB else B), transA=tA, transB=tB))
    say("gemm parts one product per output", tA, tB)
    d = normal(rng, (K,))
    want = d.astype(np.float64)[:, None] * B
    off = np.abs(product(np.diag(d)) - want)
    assert (off <= (2.0 ** -23 + 2.0 ** -24 + 2.0 ** -31) * np.abs(want)).all()
    A = np.zeros((M, K), np.float32)
    A[np.arange(M), perm] = np.exp2(rng.integers(-20, 20, M)).astype(np.float32) * \
        rng.choice([-1, 1], M).astype(np.float32)
    assert np.array_equal(product(A), A[np.arange(M), perm][:, None] * B[perm])
