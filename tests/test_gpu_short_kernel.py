"""The short-K cross-GEMM kernel against the oracle at the edges of its tiles (128
x 128 to 64 x 32) and of its 128-byte stages, and where the planner takes it: int8
and integer-valued float slices bit for bit."""
import ctypes

import pytest
import torch

from tests.helpers import assert_bitwise_equal, int_valued_slices, to_np

pytestmark = pytest.mark.gpu

FORMS = [(1, "all"), (2, "all"), (2, "triangular"), (3, "triangular"), (4, "all"),
         (4, "triangular"), (5, "triangular")]


@pytest.mark.parametrize("sdt", [torch.int8, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L,pairs", FORMS)
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (64, 32, 64), (65, 33, 128), (63, 129, 129),
                                   (128, 65, 300), (130, 31, 16), (40, 200, 63)])
def test_short_kernel(oracle, gpu, M, N, K, L, pairs, sdt):
    import ozaki_triton_amd as ozk
    from ozaki_triton_amd import _lib
    g = torch.Generator().manual_seed(1000 * L + M + N + K)
    vmax = 127 if sdt == torch.int8 else 32
    As, BsT, sa, sb = int_valued_slices(g, 2, L, M, N, K, sdt, vmax=vmax)
    for out, name in ((torch.float64, "float64"), (torch.float32, "float32")):
        with _lib.forced_kernels(gemm="short"):
            C = to_np(ozk.cross_gemm(As.to(gpu), BsT.to(gpu).transpose(-1, -2), sa.to(gpu),
                                     sb.to(gpu), L, out, pairs=pairs))
        for b in range(2):
            want = oracle.cross_gemm(to_np(As[b]), to_np(BsT[b]), to_np(sa[b]), to_np(sb[b]),
                                     name, pairs=pairs)
            assert_bitwise_equal(C[b], want, f"short L{L} {pairs} {sdt} {out} b{b}")


@pytest.mark.parametrize("sdt", [torch.int8, torch.float16])
@pytest.mark.parametrize("L,pairs,M,N", [(1, "all", 2900, 2900), (2, "all", 2100, 1000),
                                         (2, "triangular", 1000, 2100), (3, "triangular", 520, 700),
                                         (4, "all", 530, 700), (4, "triangular", 1100, 1000),
                                         (5, "triangular", 530, 300)])
def test_planner_takes_the_short_kernel(gpu, L, pairs, M, N, sdt):
    """Ragged grids just above the planner's limits: the short-K kernel by
    default, C bit for bit that of the LDS-DMA (5 slices: one-wave-per-SIMD)
    kernel."""
    import ozaki_triton_amd as ozk
    from ozaki_triton_amd import _lib
    K = 200
    g = torch.Generator().manual_seed(L + M)
    As, BsT, sa, sb = int_valued_slices(g, 1, L, M, N, K, sdt)
    args = (As.to(gpu), BsT.to(gpu).transpose(-1, -2), sa.to(gpu), sb.to(gpu), L)
    kind, ks = ctypes.c_char_p(), ctypes.c_int()
    _lib.check("ozk_debug_gemm_kernel_pairs", _lib.load().ozk_debug_gemm_kernel_pairs(
        1, M, N, K, L, {torch.int8: _lib.OZK_I8, torch.float16: _lib.OZK_F16}[sdt],
        _lib.OZK_PAIRS_TRIANGULAR if pairs == "triangular" else _lib.OZK_PAIRS_ALL, 0,
        ctypes.byref(kind), ctypes.byref(ks)))
    assert (kind.value, ks.value) == (b"short", 1)
    got = ozk.cross_gemm(*args, torch.float64, pairs=pairs)
    with _lib.forced_kernels(gemm="solo" if L == 5 else "dma"):
        want = ozk.cross_gemm(*args, torch.float64, pairs=pairs)
    assert_bitwise_equal(to_np(got), to_np(want), f"L{L} {pairs} {sdt}")


@pytest.mark.parametrize("sdt", [torch.int8, torch.float16, torch.bfloat16])
def test_one_slice_long_k(gpu, sdt):
    """One round of 128 x 128 tiles over more than 16 KB of K into fp32: the LDS-DMA
    kernel, C bit for bit that of the short-K kernel."""
    import ozaki_triton_amd as ozk
    from ozaki_triton_amd import _lib
    M, N, K = 4000, 2000, 16385 if sdt == torch.int8 else 8200
    g = torch.Generator(device=gpu).manual_seed(K)
    A = torch.randint(-32, 33, (1, 1, M, K), generator=g, device=gpu).to(sdt)
    B = torch.randint(-32, 33, (1, 1, N, K), generator=g, device=gpu).to(sdt)
    sa, sb = torch.full((1, 1, M), 0.5, device=gpu), torch.full((1, 1, N), 2.0, device=gpu)
    kind, ks = ctypes.c_char_p(), ctypes.c_int()
    assert _lib.load().ozk_debug_gemm_kernel_out(
        1, M, N, K, 1, {torch.int8: _lib.OZK_I8, torch.float16: _lib.OZK_F16,
                        torch.bfloat16: _lib.OZK_BF16}[sdt], 0, _lib.OZK_F32, 0,
        ctypes.byref(kind), ctypes.byref(ks)) == 0
    assert kind.value == b"dma"
    args = (A, B.transpose(-1, -2), sa, sb, 1, torch.float32)
    got = ozk.cross_gemm(*args)
    with _lib.forced_kernels(gemm="short"):
        want = ozk.cross_gemm(*args)
    assert_bitwise_equal(to_np(got), to_np(want), str(sdt))
