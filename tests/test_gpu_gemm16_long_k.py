"""16-bit products of few outputs and long k: summed in slices, so that no accumulator takes more
than about 1024 products.  Bar: a slice is a chain of at most 64 matrix instructions of 32 k, each
rounding (to one side, so up to 2^-23) a partial sum that grows as its square root, at most
2^-23 sqrt(64 / 2) / 2 relative to the slice's own size; slices are independent, so the whole
sum's relative error is no larger.  (In one chain per wave, K / 128 instructions: twice that.)"""
import pytest

from tests.gpu_util import require_gpu, say
from tests.routes import gemm_kernel

pytestmark = pytest.mark.gpu

BAR = 2.0 ** -23 * 32 ** 0.5 / 2     # 3.4e-7


@pytest.mark.parametrize("M,N,K", [(64, 64, 65536), (32, 32, 131072), (256, 256, 65536),
                                   (60, 100, 65530)])
@pytest.mark.parametrize("tA,tB", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("bf16", [False, True])
def test_error(M, N, K, tA, tB, bf16):
    require_gpu()
    import torch
    import cudeep_amd.ops as ops
    dt = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn((K, M) if tA else (M, K), device="cuda", generator=g).to(dt)
    b = torch.randn((N, K) if tB else (K, N), device="cuda", generator=g).to(dt)
    assert gemm_kernel("bf16" if bf16 else "f16", M, N, K, tA, tB) == "tiled"
    say("gemm16 long k", M, N, K, tA, tB, bf16)
    C = ops.gemm16(a, b, transA=tA, transB=tB).double()
    want = (a.t() if tA else a).double().contiguous() @ (b.t() if tB else b).double().contiguous()
    assert float((C - want).norm() / want.norm()) <= BAR
