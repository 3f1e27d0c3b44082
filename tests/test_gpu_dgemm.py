"""The float64 GEMM at the edges of its tiles (32 and 64 wide) and k-tiles (16), all transposes,
operands and output with their own leading dimensions."""
import numpy as np
import pytest

from tests.gpu_util import dev, host, require_gpu, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (31, 33, 15), (32, 32, 16), (33, 65, 17), (64, 64, 32),
                                   (95, 63, 33), (1025, 1023, 47), (833, 961, 49), (7, 300, 640)])
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False), (True, True)])
def test_edges(M, N, K, tA, tB):
    """Componentwise: an fp64 sum of K products in any order is within (K + 1) 2^-53 sum |a b|
    of the exact one, and so is NumPy's, against which it is held."""
    require_gpu()
    import torch
    import cudeep_amd.ops as ops
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    A = rng.standard_normal((K, M + 3) if tA else (M, K + 3))
    B = rng.standard_normal((N, K + 5) if tB else (K, N + 5))
    a, b = (A[:, 1:M + 1] if tA else A[:, 1:K + 1]), (B[:, 2:K + 2] if tB else B[:, 2:N + 2])
    dA, dB = dev(A), dev(B)
    va = dA[:, 1:M + 1] if tA else dA[:, 1:K + 1]
    vb = dB[:, 2:K + 2] if tB else dB[:, 2:N + 2]
    buf = torch.full((M + 2, N + 4), -7.0, device="cuda", dtype=torch.float64)
    say("dgemm edges", M, N, K, tA, tB)
    C = host(ops.dgemm(va, vb, tA, tB, out=buf[1:M + 1, 3:N + 3]))
    oa, ob = (a.T if tA else a), (b.T if tB else b)
    bound = 2 * (K + 1) * 2.0 ** -53 * (np.abs(oa) @ np.abs(ob))
    assert (np.abs(C - oa @ ob) <= bound).all()
    full = host(buf)
    full[1:M + 1, 3:N + 3] = -7.0
    assert (full == -7.0).all()
