"""Where the planner leaves the short-K cross-GEMM kernel (no GPU needed): one
slice over a long K where both kernels' tiles are one round, and more tiles
than one launch counts."""
import ctypes

import pytest


def _plan(M, N, K, L, sd, pairs="all", out="float64"):
    from ozaki_triton_amd import _lib
    name, ks = ctypes.c_char_p(), ctypes.c_int()
    codes = {"float64": _lib.OZK_F64, "float32": _lib.OZK_F32, "float16": _lib.OZK_F16,
             "bfloat16": _lib.OZK_BF16, "int8": _lib.OZK_I8}
    st = _lib.load().ozk_debug_gemm_kernel_out(
        1, M, N, K, L, codes[sd], int(pairs == "triangular"), codes[out], 256, ctypes.byref(name),
        ctypes.byref(ks))
    assert st == 0, _lib.strerror(st)
    return name.value.decode()


@pytest.mark.parametrize("sd,size", [("int8", 1), ("float16", 2), ("bfloat16", 2)])
def test_one_slice_over_a_long_k(sd, size):
    for M, N in ((4096, 2048), (8192, 1024), (4000, 2000)):   # 512 tiles of 128 x 128
        for out in ("float32", sd):
            assert _plan(M, N, 16384 // size, 1, sd, out=out) == "short"
            assert _plan(M, N, 16384 // size + 1, 1, sd, out=out) == "dma"
        assert _plan(M, N, 65536 // size, 1, sd) == "short"   # into fp64
    # other rounds: the LDS-DMA kernel's last one is half empty, or its tiles are more
    for M, N in ((4096, 2176), (3000, 3400), (4096, 4096)):
        assert _plan(M, N, 65536 // size, 1, sd, out="float32") == "short"
    assert _plan(2048, 2048, 256, 1, sd, out="float32") == "dma"


def test_more_tiles_than_a_launch_counts():
    """2^24 tiles of 64 x 32 are 2^32 work-items: larger tiles, which launch."""
    assert _plan(1 << 18, (1 << 17) - 32, 64, 4, "int8") == "short"
    assert _plan(1 << 18, 1 << 17, 64, 4, "int8") == "wide4"
    assert _plan(1 << 18, 1 << 17, 64, 5, "int8", "triangular") == "solo"
    assert _plan(1 << 18, 1 << 17, 64, 4, "float16", "triangular") != "short"
