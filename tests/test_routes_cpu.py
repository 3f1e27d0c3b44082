"""The kernels that the library chooses (no GPU needed): both sides of each line."""
import pytest

from tests.routes import gemm_kernel


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K,tA,tB,want", [
    (64, 64, 4096, False, False, "direct"),       # a wave sums no more than a k-slice would
    (64, 64, 4104, False, False, "tiled"),
    (64, 64, 65536, False, True, "tiled"),
    (32, 32, 131072, True, False, "tiled"),
    (192, 24, 14208, True, False, "tiled"),
    (416, 896, 8856, False, False, "tiled"),      # 98 tiles: the tiled kernel slices k
    (700, 760, 8856, False, False, "direct"),     # 132 tiles: it does not
    (512, 512, 1024, False, True, "direct"),      # whole tiles, 256 of 32 x 32
    (576, 512, 1024, False, True, "tiled"),
    (576, 512, 1024, False, False, "tiled"),
    (576, 512, 1024, True, True, "tiled"),
    (512, 640, 1024, True, False, "direct"),      # A transposed, B not: 320
    (576, 640, 1024, True, False, "tiled"),
    (600, 608, 1000, False, True, "direct"),      # ragged: 768
])
def test_gemm16(kind, M, N, K, tA, tB, want):
    assert gemm_kernel(kind, M, N, K, tA, tB) == want
