"""Which kernel the library runs for a call (its own choice, asked without a GPU)."""
import ctypes

from cudeep_amd import _lib as L


def gemm_kernel(kind, M, N, K, tA=False, tB=False, lda=None, ldb=None):
    """`kind`: a precision mode, or torch-like "bf16" / "f16" operands; 16-byte aligned
    operands with the given leading dimensions (dense by default)."""
    f = L.lib().cdxi_gemm_kernel
    f.restype, f.argtypes = ctypes.c_char_p, [ctypes.c_int] * 3 + [ctypes.c_int64] * 5
    code = {"bf16": 16 + L.DTYPE_BF16, "f16": 16 + L.DTYPE_F16}.get(kind, kind)
    return f(code, int(tA), int(tB), M, N, K, lda or (M if tA else K),
             ldb or (K if tB else N)).decode()


def conv_kernel(what, B, IC, OC, H, W, KH, KW, stride=(1, 1), pad=(0, 0)):
    """`what`: "forward", "implicit" (the implicit forward entry point) "data" or "weight"
    (backward)."""
    f = L.lib().cdxi_conv_kernel
    f.restype, f.argtypes = ctypes.c_char_p, [ctypes.c_int] + [ctypes.c_int64] * 11
    return f(("forward", "implicit", "data", "weight").index(what), B, IC, OC, H, W, KH, KW, *stride,
             *pad).decode()
