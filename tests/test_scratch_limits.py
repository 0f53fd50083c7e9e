"""Long operands that are not whole 16-byte pieces (K % 4, pitch, alignment) with
less scratch than their plan would take: they run on the generic split kernel,
in ozk_matmul_static's 64 MiB and without a workspace in ozk_split; whole
operands are refused there.  And with all they ask for: long columns are
transposed in parts of 128 MiB."""
import ctypes

import pytest
import torch

from tests.helpers import (assert_bitwise_equal, c3_like, check_block_vs_oracle,
                           oracle_split_batched, sample_indices, to_np)


# M, N, K, dtype, L: the transposed copy of B alone is 238 and 66 MB; A's rows of
# the third are cut along K
RAGGED = [(100, 900, 33001, "float64", 1), (64, 1000, 16389, "float32", 1),
          (300, 20, 40003, "float32", 4)]


def _need(lib, code, M, N, K, L, have):
    from ozaki_triton_amd import _lib
    nb = ctypes.c_size_t(0)
    st = lib.ozk_debug_matmul_workspace(code, 1, M, N, K, _lib.i64arr([0, K, 1]),
                                        _lib.i64arr([0, N, 1]), L, _lib.OZK_I8, have,
                                        ctypes.byref(nb))
    assert st == 0, _lib.strerror(st)
    return nb.value


@pytest.mark.parametrize("M,N,K,xdt,L", RAGGED)
def test_ragged_long_k_needs_only_its_slices(M, N, K, xdt, L):
    from ozaki_triton_amd import _lib
    lib = _lib.load()
    code = {"float64": _lib.OZK_F64, "float32": _lib.OZK_F32}[xdt]
    kp = (K + 15) // 16 * 16
    slices = sum((x + 255) // 256 * 256 for x in (L * M * kp, L * M * 4, L * N * kp, L * N * 4))
    assert _need(lib, code, M, N, K, L, 0) == slices <= _lib.OZK_STATIC_SCRATCH_BYTES
    whole = _need(lib, code, M, N, K, L, 1 << 62)
    assert whole > slices
    # exactly enough: the planner's own choice
    assert _need(lib, code, M, N, K, L, whole) == whole
    # a whole K needs its scratch, whatever there is
    Kw = (K + 15) // 16 * 16
    assert _need(lib, code, M, N, Kw, L, 0) == _need(lib, code, M, N, Kw, L, 1 << 62) > slices


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,xdt,L", RAGGED)
def test_static_runs_ragged_long_k(oracle, gpu, M, N, K, xdt, L):
    import ozaki_triton_amd as ozk
    from ozaki_triton_amd import _lib
    lib = _lib.load()
    dt = getattr(torch, xdt)
    A, B = c3_like((M, K), (K, N), seed=K, dtype=dt)
    Ad, Bd = A.to(gpu), B.to(gpu)
    C = torch.full((M, N), float("nan"), dtype=dt, device=gpu)
    print(f"[static] {M}x{N}x{K} {xdt} L={L}", flush=True)
    st = lib.ozk_matmul_static(
        ctypes.c_void_p(Ad.data_ptr()), _lib.i64arr([0, K, 1]), ctypes.c_void_p(Bd.data_ptr()),
        _lib.i64arr([0, N, 1]), _lib.OZK_F64 if xdt == "float64" else _lib.OZK_F32, 1, M, N, K, L,
        _lib.OZK_I8, ctypes.c_void_p(C.data_ptr()), _lib.i64arr([0, N, 1]), None,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0, _lib.strerror(st)
    want = ozk.ozaki_matmul(Ad, Bd, L, torch.int8)
    torch.cuda.synchronize()
    assert_bitwise_equal(to_np(C), to_np(want), "static vs the planner's own kernels")
    check_block_vs_oracle(oracle, ozk, to_np(C), to_np(A), to_np(B), sample_indices(M, 6, 1),
                          sample_indices(N, 6, 2), L, torch.int8, dt, "static vs oracle")


@pytest.mark.gpu
@pytest.mark.parametrize("xdt", [torch.float64, torch.float32])
@pytest.mark.parametrize("columns,rows,K", [(True, 37, 33001), (True, 18, 16387), (False, 5, 20001)])
def test_split_without_a_workspace(oracle, gpu, columns, rows, K, xdt):
    """ozk_split on a ragged operand with no workspace at all: the oracle's bits; a
    whole operand of the same kind is refused."""
    from ozaki_triton_amd import _lib
    lib = _lib.load()
    L, alpha = 2, 7
    g = torch.Generator().manual_seed(K)
    for k, ok in ((K, True), ((K + 15) // 16 * 16, False)):
        X = torch.randn(1, rows, k, generator=g, dtype=torch.float64).to(xdt)
        Xd = X.to(gpu).mT.contiguous().mT if columns else X.to(gpu)
        sl = torch.zeros(1, L, rows, k, dtype=torch.int8, device=gpu)
        sc = torch.zeros(1, L, rows, dtype=torch.float32, device=gpu)
        st = lib.ozk_split(
            ctypes.c_void_p(Xd.data_ptr()),
            _lib.OZK_F64 if xdt == torch.float64 else _lib.OZK_F32, 1, rows, k,
            _lib.i64arr(Xd.stride()), L, alpha, _lib.OZK_I8, ctypes.c_void_p(sl.data_ptr()),
            _lib.i64arr(sl.stride()), ctypes.c_void_p(sc.data_ptr()), _lib.i64arr(sc.stride()),
            None, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        if not ok:
            assert st == _lib.OZK_ERR_WORKSPACE
            continue
        assert st == 0, _lib.strerror(st)
        osl, osc = oracle_split_batched(oracle, to_np(X), L, alpha, torch.int8)
        assert_bitwise_equal(to_np(sc), osc, "scales")
        assert_bitwise_equal(to_np(sl), osl, "slices")


# batch, rows (columns of the operand in memory), K, dtype: several parts of
# 128 MiB, of one batch's rows (the last part short) and of whole batches
PARTS = [(1, 1100, 33001, "float64"), (2, 513, 33003, "float64"), (37, 100, 16387, "float32")]


def _split_bytes(lib, batch, rows, K, xdt, L):
    from ozaki_triton_amd import _lib
    nb = ctypes.c_size_t(0)
    st = lib.ozk_split_workspace_bytes(
        _lib.OZK_F64 if xdt == "float64" else _lib.OZK_F32, batch, rows, K,
        _lib.i64arr([rows * K, 1, rows]), L, _lib.OZK_I8,
        _lib.i64arr([L * rows * K, rows * K, K, 1]), ctypes.byref(nb))
    assert st == 0
    return nb.value


@pytest.mark.parametrize("batch,rows,K,xdt", PARTS + [(4, 16384, 65537, "float64")])
def test_transposed_parts_are_bounded(batch, rows, K, xdt):
    from ozaki_triton_amd import _lib
    got = _split_bytes(_lib.load(), batch, rows, K, xdt, 1)
    assert 64 << 20 < got <= 130 << 20 < batch * rows * K * (8 if xdt == "float64" else 4)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,rows,K,xdt", PARTS)
def test_split_transposed_in_parts(oracle, gpu, force, batch, rows, K, xdt):
    import ozaki_triton_amd as ozk
    from ozaki_triton_amd import _lib
    L, alpha = 2, 7
    print(f"[parts] {batch}x{rows}x{K} {xdt}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(K)
    Xd = torch.randn(batch, K, rows, generator=g, dtype=getattr(torch, xdt), device=gpu).mT
    sl, sc = ozk.split_matrix(Xd, L, alpha, torch.int8)
    force(split="generic")
    gsl, gsc = ozk.split_matrix(Xd, L, alpha, torch.int8)
    torch.cuda.synchronize()
    assert torch.equal(sc, gsc) and torch.equal(sl, gsl)
    for b in (0, batch - 1):
        idx = torch.tensor([0, rows // 2, rows - 1], device=gpu)
        osl, osc = oracle_split_batched(oracle, to_np(Xd[b:b + 1, idx].contiguous()), L, alpha,
                                        torch.int8)
        assert_bitwise_equal(to_np(sc[b:b + 1, :, idx].contiguous()), osc, "scales")
        assert_bitwise_equal(to_np(sl[b:b + 1, :, idx].contiguous()), osl, "slices")
    # waits that give up: every part's scales are NaN, the device status is set
    force(split="", coop_timeout=True)
    ozk.device_status()
    sl, sc = ozk.split_matrix(Xd, L, alpha, torch.int8)
    torch.cuda.synchronize()
    assert torch.isnan(sc).all()
    with pytest.raises(_lib.OzakiLibError):
        ozk.device_status()
