"""The split kernels at K that is no multiple of 4 (or of a 16-byte slice
piece), rows and columns of any alignment, column counts that leave a group
part empty, and narrow inputs converted as they are loaded: slices and scales
bit for bit against the oracle, and ozaki_matmul's zero-padded slice rows
against the cross-GEMM of packed ones."""
import pytest
import torch

from tests.helpers import (assert_bitwise_equal, check_block_vs_oracle, oracle_split_batched,
                           sample_indices, to_np)

pytestmark = pytest.mark.gpu

INPUTS = [torch.float64, torch.float32, torch.float16, torch.bfloat16, torch.int8]


def _operand(g, batch, rows, K, dtype):
    if dtype == torch.int8:
        return torch.randint(-128, 128, (batch, rows, K), generator=g, dtype=torch.int8)
    X = torch.randn(batch, rows, K, generator=g, dtype=torch.float64)
    return (X * torch.pow(2.0, torch.randint(-3, 4, (batch, rows, 1), generator=g).double())).to(dtype)


# (rows, K): either side of each class's limit, one element, a last group of
# columns part full, long rows (shared by workgroups) and columns
# (cooperative, transposed)
SIZES = [(5, 1), (9, 3), (7, 255), (33, 257), (130, 511), (21, 515), (40, 1023), (2051, 1027),
         (19, 2047), (4099, 2049), (11, 4095), (2053, 4095), (6, 4097), (2049, 4101), (3, 8191)]
LONG = [(5, 8193), (18, 16383), (3, 16387), (7, 33001), (5, 65533)]


@pytest.mark.parametrize("columns", [False, True])
@pytest.mark.parametrize("xdt", INPUTS)
@pytest.mark.parametrize("rows,K", SIZES + LONG)
def test_split_ragged(oracle, gpu, rows, K, xdt, columns):
    import ozaki_triton_amd as ozk
    sdt = [torch.int8, torch.float16, torch.bfloat16, torch.float32][(rows + K) % 4]
    L, batch = 1 + K % 4, 2 if rows * K < 1 << 20 else 1
    print(f"[ragged] {rows}x{K} {xdt} -> {sdt} L={L} columns={columns}", flush=True)
    g = torch.Generator().manual_seed(rows * 31 + K)
    X = _operand(g, batch, rows, K, xdt)
    Xd = X.to(gpu)
    if columns:   # the B^T view, one element past an aligned address
        buf = torch.empty(1 + X.numel(), dtype=xdt, device=gpu)[1:].view(batch, K, rows)
        buf.copy_(Xd.mT)
        Xd = buf.mT
    alpha = ozk.compute_split_bits(
        K, sdt, torch.int32 if sdt == torch.int8 else torch.float32)
    sl, sc = ozk.split_matrix(Xd, L, alpha, sdt)
    torch.cuda.synchronize()
    # the oracle on sampled rows (the split is per row)
    idx = sample_indices(rows, min(rows, 24), K)
    osl, osc = oracle_split_batched(oracle, to_np(X[:, idx].contiguous()), L, alpha, sdt)
    assert_bitwise_equal(to_np(sc[:, :, idx].contiguous()), osc, "scales")
    assert_bitwise_equal(to_np(sl[:, :, idx].contiguous()), osl, "slices")


@pytest.mark.parametrize("sdt", [torch.int8, torch.float16])
@pytest.mark.parametrize("xdt", INPUTS)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("M,N,K", [(65, 97, 257), (130, 70, 1001), (40, 2050, 4103)])
def test_matmul_ragged_layouts(oracle, gpu, M, N, K, ta, tb, xdt, sdt):
    """Both operands by split_fused_kernel (or, with wide column groups, in two
    launches) in every layout, into zero-padded slice rows."""
    import ozaki_triton_amd as ozk
    g = torch.Generator().manual_seed(M + N + K)
    A, B = _operand(g, 1, M, K, xdt)[0], _operand(g, 1, N, K, xdt)[0].T.contiguous()
    Ad = A.T.contiguous().to(gpu).T if ta else A.to(gpu)
    Bd = B.T.contiguous().to(gpu).T if tb else B.to(gpu)
    C = ozk.ozaki_matmul(Ad, Bd, 3, sdt)
    torch.cuda.synchronize()
    if xdt == torch.int8 and sdt != torch.int8:
        # a truncated int8 C of float slices: no bound to check it with, but the
        # slices split alone, packed for the cross-GEMM, give the same bits
        alpha = ozk.compute_split_bits(K, sdt, torch.float32)
        a_sl, a_sc = ozk.split_matrix(Ad.unsqueeze(0), 3, alpha, sdt)
        b_sl, b_sc = ozk.split_matrix(Bd.T.unsqueeze(0), 3, alpha, sdt)
        want = ozk.cross_gemm(a_sl, b_sl.transpose(-1, -2), a_sc, b_sc, 3, xdt)[0]
        assert_bitwise_equal(to_np(C), to_np(want), f"{ta} {tb}")
        return
    check_block_vs_oracle(oracle, ozk, to_np(C), to_np(A), to_np(B), sample_indices(M, 16, 1),
                          sample_indices(N, 16, 2), 3, sdt, xdt, f"{ta} {tb}")


@pytest.mark.parametrize("sdt", [torch.int8, torch.float16])
def test_matmul_ragged_infinite_row(gpu, sdt):
    """A row of A with an infinite entry spoils its row of C only: the padding
    of its slice rows is zero, whatever the row's scale."""
    import ozaki_triton_amd as ozk
    g = torch.Generator().manual_seed(3)
    A, B = _operand(g, 1, 70, 515, torch.float32)[0], _operand(g, 1, 515, 66, torch.float32)[0]
    want = ozk.ozaki_matmul(A.to(gpu), B.to(gpu), 3, sdt)
    A[9, 514] = float("inf")
    got = ozk.ozaki_matmul(A.to(gpu), B.to(gpu), 3, sdt)
    torch.cuda.synchronize()
    keep = [i for i in range(70) if i != 9]
    assert not torch.isfinite(got[9]).any()
    assert_bitwise_equal(to_np(got[keep]), to_np(want[keep]), "other rows")
