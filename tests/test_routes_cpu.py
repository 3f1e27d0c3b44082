"""The kernels that the library chooses (no GPU needed): both sides of each line."""
import pytest

from cudeep_amd import _lib as L
from tests.routes import conv_kernel, gemm_kernel


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


@pytest.mark.parametrize("M,N,K,tA,tB,want", [
    (2048, 2048, 48, False, False, "tiled"),      # short k: the pipeline only fills
    (2048, 2048, 128, False, False, "parts"),
    (5104, 716, 64, True, True, "tiled"),
    (4096, 4096, 48, False, True, "tiled"),
    (4096, 4096, 512, False, True, "parts"),
    (25088, 392, 32, False, False, "tiled"),
    (2048, 2304, 64, False, False, "tiled"),      # 288 tiles: a second round of 32
    (2048, 2304, 2048, False, False, "parts"),
    (2048, 2304, 2048, True, False, "tiled"),
    (2999, 1501, 2048, True, False, "parts"),     # rows the tiled kernel reads one by one
    (8192, 784, 256, False, False, "parts"),
    (4096, 4096, 4096, True, True, "parts"),
    (256, 785, 8192, True, False, "parts"),       # k-slices
])
def test_gemm_f32_parts(M, N, K, tA, tB, want):
    assert gemm_kernel(0, M, N, K, tA, tB) == want


@pytest.mark.parametrize("M,N,K,tA,tB,want", [
    (640, 640, 512, False, False, "direct"),      # up to 400 tiles of 32 x 32
    (640, 672, 512, False, False, "tiled"),
    (1200, 1200, 100, True, False, "direct"),     # only k ragged: 1450 tiles
    (1600, 1600, 300, False, True, "tiled"),
    (16896, 84, 1564, False, True, "direct"),     # NT, long k: 2200
    (1301, 1301, 90, True, False, "direct"),      # rows ragged: 1700
    (1601, 1601, 61, False, False, "direct"),     # beyond, by k and orientation
    (1601, 1601, 61, False, True, "direct"),
    (1601, 1601, 65, False, True, "tiled"),
    (1601, 1601, 701, False, True, "direct"),
    (1368, 1664, 153, True, True, "direct"),
    (1369, 1664, 152, True, True, "tiled"),
    (1401, 1451, 701, True, False, "direct"),     # 2024 tiles
    (1601, 1601, 701, True, False, "tiled"),      # 2601
    (61, 100001, 301, False, False, "tiled"),     # one side within 64: wide tiles there
    (100001, 61, 301, False, True, "tiled"),
    (548, 4441, 120, False, False, "direct"),
    (548, 4441, 20, False, False, "tiled"),
    (14912, 196, 2302, False, False, "direct"),
    (90, 50001, 301, False, True, "tiled"),       # more than 4096 tiles
    (90, 40001, 101, False, False, "tiled"),      # more than 3000
])
def test_gemm_f32_direct(M, N, K, tA, tB, want):
    assert gemm_kernel(0, M, N, K, tA, tB) == want


# B, IC, OC, H, W, KH, KW, stride, padding
@pytest.mark.parametrize("g,want", [
    ((6, 56, 46, 31, 31, 3, 3, (2, 2), (1, 1)), "direct"),       # below 4 MiB of columns
    ((3, 168, 99, 56, 56, 1, 1, (2, 2), (0, 0)), "direct"),
    ((1, 160, 64, 28, 28, 5, 5, (2, 2), (2, 2)), "direct"),      # 4000 k
    ((1, 161, 64, 28, 28, 5, 5, (2, 2), (2, 2)), "im2col"),
    ((2, 200, 48, 14, 14, 7, 7, (2, 2), (3, 3)), "im2col"),
    ((4, 256, 512, 56, 56, 1, 1, (2, 2), (0, 0)), "im2col"),     # row-window tiles enough, but 1x1
    ((7, 4, 200, 60, 60, 3, 3, (2, 2), (1, 1)), "rowwin"),       # k < 128
    ((16, 14, 128, 112, 112, 1, 1, (2, 2), (0, 0)), "rowwin"),   # 1x1 of 14 channels
    ((1, 128, 168, 13, 13, 11, 11, (4, 4), (5, 5)), "im2col"),   # more taps than a mask holds
    ((16, 3, 64, 224, 224, 7, 7, (2, 2), (3, 3)), "gather"),     # beyond 4 MiB
    ((2, 16, 16, 12, 12, 3, 3, (1, 1), (1, 1)), "im2col"),       # the Winograd shape
    ((16, 256, 64, 56, 56, 1, 1, (1, 1), (0, 0)), "product"),
    ((1, 16, 176, 7, 7, 1, 1), "direct"),                        # one image, 16 k, few pixels
    ((1, 8, 40, 31, 31, 1, 1), "product"),                       # (no im2col for it)
    ((1, 9, 512, 56, 56, 1, 1), "product"),
    ((1, 17, 176, 7, 7, 1, 1), "product"),
    ((1, 12, 40, 13, 13, 11, 11, (4, 4), (5, 5)), "im2col"),
])
def test_conv_forward(g, want):
    assert conv_kernel("forward", *g) == want


@pytest.mark.parametrize("g,want", [
    ((2, 12, 512, 28, 28, 3, 3, (1, 1), (1, 1)), "rowwin"),      # k < 128, 64-channel waves
    ((16, 3, 64, 56, 56, 5, 5, (2, 2), (2, 2)), "rowwin"),
    ((4, 12, 96, 31, 31, 3, 3, (2, 2), (1, 1)), "direct"),       # 32-channel waves
    ((4, 96, 100, 56, 56, 1, 1, (2, 2), (0, 0)), "direct"),      # 1x1 with a stride
    ((2, 15, 512, 28, 28, 3, 3, (1, 1), (1, 1)), "direct"),      # k = 135
    ((16, 8, 51, 28, 28, 7, 7, (1, 1), (3, 3)), "rowwin"),       # eight channels, 112 tiles
    ((16, 9, 51, 28, 28, 7, 7, (1, 1), (3, 3)), "direct"),
    ((16, 6, 24, 31, 31, 7, 7, (1, 1), (3, 3)), "direct"),       # (pads less)
    ((6, 4, 129, 56, 56, 7, 7, (2, 2), (3, 3)), "rowwin"),
    ((9, 4, 64, 14, 14, 5, 5, (1, 1), (2, 2)), "rowwin"),        # four channels
    ((9, 5, 64, 14, 14, 5, 5, (1, 1), (2, 2)), "direct"),
    ((8, 3, 64, 31, 31, 7, 7, (2, 2), (3, 3)), "direct"),
    ((2, 16, 168, 224, 224, 7, 7, (2, 2), (3, 3)), "gather"),    # 2352 tiles
    ((9, 80, 81, 112, 112, 7, 7, (2, 2), (3, 3)), "direct"),     # (pads less)
    ((8, 64, 128, 112, 112, 7, 7, (2, 2), (3, 3)), "direct"),    # 1568
    ((8, 8, 127, 112, 112, 7, 7, (2, 2), (3, 3)), "gather"),     # eight channels
])
def test_conv_implicit(g, want):
    assert conv_kernel("implicit", *g) == want


@pytest.mark.parametrize("g,want", [
    ((2, 256, 8, 28, 28, 3, 3, (1, 1), (1, 1)), "rowwin"),       # k = 72
    ((2, 256, 15, 28, 28, 3, 3, (1, 1), (1, 1)), "direct"),      # k = 135
    ((98, 12, 64, 16, 16, 3, 3, (1, 1), (1, 1)), "direct"),      # 12 channels
    ((1, 2048, 8, 13, 13, 1, 1), "direct"),                      # 1x1: few to many channels
    ((2, 2048, 8, 13, 13, 1, 1), "product"),
    ((1, 32, 16, 224, 224, 1, 1), "product"),
    ((1, 3, 8, 31, 31, 1, 1), "direct"),
    ((1, 3, 8, 28, 28, 1, 1), "product"),
    ((1, 64, 2048, 20, 20, 1, 1), "direct"),                     # k-slices
])
def test_conv_backward_data(g, want):
    assert conv_kernel("data", *g) == want


@pytest.mark.parametrize("g,want", [
    ((64, 512, 512, 28, 28, 1, 1), "direct"),                        # 1x1
    ((32, 1024, 1024, 14, 14, 3, 3, (1, 1), (1, 1)), "direct"),      # rows of up to 16
    ((4, 64, 64, 28, 28, 3, 3, (1, 1), (1, 1)), "direct"),           # 504 workgroups
    ((16, 16, 128, 28, 28, 3, 3, (1, 1), (1, 1)), "rows"),           # 1120
    ((8, 128, 16, 40, 40, 3, 3, (1, 1), (1, 1)), "direct"),          # rows of 40 in 56
    ((16, 8, 16, 112, 112, 3, 3, (1, 1), (1, 1)), "direct"),         # mostly padding
    ((32, 64, 64, 56, 56, 3, 3, (1, 1), (1, 1)), "rows"),            # 7 GFLOP
    ((4, 128, 128, 28, 28, 3, 3, (2, 2), (1, 1)), "direct"),         # 36 workgroups
    ((32, 32, 192, 31, 31, 3, 3, (2, 2), (1, 1)), "gather"),         # 192
    ((16, 16, 32, 112, 112, 5, 5, (1, 1), (2, 2)), "direct"),        # padding
    ((16, 200, 72, 7, 7, 5, 5, (2, 2), (2, 2)), "direct"),
    ((1, 227, 120, 13, 13, 7, 7, (2, 2), (3, 3)), "gather"),         # one step per wave
    ((1, 204, 136, 7, 7, 5, 5, (2, 2), (2, 2)), "direct"),
    ((16, 200, 144, 31, 31, 3, 3, (2, 2), (1, 1)), "gather"),
    ((8, 158, 138, 112, 112, 1, 1, (2, 2), (0, 0)), "gather"),       # 1x1 with a stride
    ((64, 200, 168, 56, 56, 1, 1, (2, 2), (0, 0)), "direct"),
    ((16, 48, 48, 28, 28, 1, 1, (2, 2), (0, 0)), "direct"),
    ((8, 177, 256, 7, 7, 5, 5, (2, 2), (2, 2)), "direct"),           # two steps per wave
    ((20, 128, 168, 28, 28, 7, 7, (2, 2), (3, 3)), "direct"),        # 198
    ((16, 24, 56, 224, 224, 5, 5, (1, 1), (2, 2)), "direct"),        # 196 steps per wave
    ((1, 512, 512, 14, 14, 3, 3, (2, 2), (1, 1)), "gather"),         # one
    ((16, 3, 64, 224, 224, 7, 7, (2, 2), (3, 3)), "gather"),         # whole channels, 4 GFLOP
])
def test_conv_backward_weight(g, want):
    assert conv_kernel("weight", *g) == want


@pytest.mark.parametrize("g,want", [((1, 16, 128, 7, 7), 1), ((1, 14, 128, 7, 7), 0),
                                    ((4, 128, 128, 28, 28), 1), ((8, 64, 64, 56, 56), 0),
                                    ((2, 256, 64, 20, 20), 1), ((2, 257, 64, 20, 20), 0),
                                    ((3, 512, 48, 20, 20), 0)])
def test_small_3x3(g, want):
    from cudeep_amd import _lib as L
    assert L.lib().cdx_conv2d_3x3_is_small(*g) == want


@pytest.mark.parametrize("g", [(1, 161, 14, 15, 5, 5, (2, 2), (2, 2)), (2, 82, 9, 9, 7, 7, (2, 2), (3, 3)),
                               (1, 40, 13, 13, 11, 11, (4, 4), (5, 5)), (1, 4100, 9, 8, 1, 1, (1, 1), (0, 0))])
def test_columns_of_a_long_k_have_room_for_slices(g):
    """The forward query covers the column buffer and the slices of the columns' product, for any
    number of output channels."""
    lib = L.lib()
    B, IC, H, W, KH, KW, (sh, sw), (ph, pw) = g
    K, ns = IC * KH * KW, B * ((H + 2 * ph - KH) // sh + 1) * ((W + 2 * pw - KW) // sw + 1)
    got = lib.cdx_conv2d_forward_workspace_size(B, IC, H, W, KH, KW, sh, sw, ph, pw)
    tiles_n, most = -(-ns // 64), 0
    for OC in range(17, 64 * (127 // tiles_n) + 1):
        assert conv_kernel("forward", B, IC, OC, H, W, KH, KW, (sh, sw), (ph, pw)) == "im2col"
        if lib.cdx_gemm_workspace_size(0, 0, 0, OC, ns, K) > 0:
            # (64-row tiles, 128 x 64 from 128 rows on; about 768 slices of tiles of 256 k or more)
            tiles = -(-OC // (128 if OC >= 128 else 64)) * tiles_n
            s = min((768 + tiles // 2) // tiles, K // 256)
            chunk = -(-(-(-K // s)) // 16) * 16
            most = max(most, -(-K // chunk) * OC * ns * 4)
    assert most > 0 and got >= 4 * K * ns + 255 + most


@pytest.mark.parametrize("g", [(1, 160, 28, 28, 5, 5, (2, 2), (2, 2)), (2, 3, 9, 9, 3, 3, (1, 1), (1, 1)),
                               (2, 5000, 5, 5, 1, 1, (1, 1), (0, 0))])
def test_other_layers_ask_for_columns_only(g):
    B, IC, H, W, KH, KW, (sh, sw), (ph, pw) = g
    ns = B * ((H + 2 * ph - KH) // sh + 1) * ((W + 2 * pw - KW) // sw + 1)
    assert L.lib().cdx_conv2d_forward_workspace_size(B, IC, H, W, KH, KW, sh, sw, ph, pw) \
        == 4 * IC * KH * KW * ns
