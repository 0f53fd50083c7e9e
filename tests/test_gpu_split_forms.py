"""The three forms of the split kernels (exact sizes, whole quads, any): slices and
scales bit for bit against the oracle in every class of K, rows and columns,
and ozaki_matmul's zero padding of whole quads beside a row with an infinite
entry."""
import pytest
import torch

from tests.helpers import assert_bitwise_equal, oracle_split_batched, sample_indices, to_np

pytestmark = pytest.mark.gpu

SDTS = [torch.int8, torch.float16, torch.bfloat16, torch.float32]
# (rows, K): K at a class's limit with whole groups; whole quads and groups of
# columns part empty; the same with wide column groups (fp64 from 256 groups of 8
# columns at K <= 1024, 512 at K <= 2048, fp64 and fp32 256 of 4 and 8 at K <= 4096)
EXACT = [(16, 256), (16, 512), (8, 1024), (8, 2048), (8, 4096), (8, 8192), (8, 16384)]
WHOLE = [(20, 100), (12, 300), (36, 516), (12, 1028), (28, 2052), (12, 4100), (8, 8196), (12, 12292)]
WIDE = [(2048, 1024), (2060, 1020), (2053, 1021), (2049, 700), (4096, 2048), (4108, 2044),
        (4099, 2045), (4097, 1500), (2048, 4096), (2060, 4092)]


@pytest.mark.parametrize("xdt", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("columns,rows,K", [(False, *s) for s in EXACT + WHOLE] +
                         [(True, *s) for s in EXACT + WHOLE + WIDE])
def test_split_forms(oracle, gpu, columns, rows, K, xdt):
    import ozaki_triton_amd as ozk
    sdt = SDTS[(rows // 4 + K // 4 + (xdt == torch.float32)) % 4]
    L, batch = 1 + (rows + K // 4) % 4, 2 if rows * K < 1 << 20 else 1
    print(f"[forms] {rows}x{K} {xdt} -> {sdt} L={L} columns={columns}", flush=True)
    g = torch.Generator().manual_seed(rows * 17 + K)
    X = torch.randn(batch, rows, K, generator=g, dtype=torch.float64)
    X = (X * torch.pow(2.0, torch.randint(-3, 4, (batch, rows, 1), generator=g).double())).to(xdt)
    Xd = X.to(gpu)
    if columns:
        Xd = Xd.mT.contiguous().mT
    alpha = ozk.compute_split_bits(K, sdt, torch.int32 if sdt == torch.int8 else torch.float32)
    sl, sc = ozk.split_matrix(Xd, L, alpha, sdt)
    torch.cuda.synchronize()
    idx = sample_indices(rows, min(rows, 24), K)
    osl, osc = oracle_split_batched(oracle, to_np(X[:, idx].contiguous()), L, alpha, sdt)
    assert_bitwise_equal(to_np(sc[:, :, idx].contiguous()), osc, "scales")
    assert_bitwise_equal(to_np(sl[:, :, idx].contiguous()), osl, "slices")


@pytest.mark.parametrize("sdt", SDTS)
@pytest.mark.parametrize("xdt", [torch.float64, torch.float32])
@pytest.mark.parametrize("M,N,K", [(72, 68, 516), (40, 36, 1028)])
def test_whole_quads_infinite_entries(gpu, M, N, K, xdt, sdt):
    """Infinite entries spoil their row and column of C only: the quads of padding
    after a K of whole quads stay zero, whatever the scale."""
    import ozaki_triton_amd as ozk
    g = torch.Generator().manual_seed(K)
    A = torch.randn(M, K, generator=g, dtype=torch.float64).to(xdt)
    B = torch.randn(K, N, generator=g, dtype=torch.float64).to(xdt)
    want = ozk.ozaki_matmul(A.to(gpu), B.to(gpu), 3, sdt)
    A[9, K - 1] = float("inf")
    B[0, 5] = float("-inf")
    got = ozk.ozaki_matmul(A.to(gpu), B.to(gpu), 3, sdt)
    torch.cuda.synchronize()
    assert not torch.isfinite(got[9]).any() and not torch.isfinite(got[:, 5]).any()
    rows, cols = [i for i in range(M) if i != 9], [j for j in range(N) if j != 5]
    assert_bitwise_equal(to_np(got[rows][:, cols]), to_np(want[rows][:, cols]), "other entries")


# batches of 1, 2, prime, a power of two and one more or less rows (the row's batch
# is a multiplication), and workgroups of 1 and 4 rows that cross batches
@pytest.mark.parametrize("batch,rows", [(1, 9), (9, 1), (5, 2), (6, 3), (3, 7), (4, 8), (3, 17), (2, 31),
                                        (3, 127), (3, 257)])
@pytest.mark.parametrize("K", [60, 192, 320, 703, 704, 1344, 2900])
def test_batched_rows(oracle, gpu, batch, rows, K):
    import ozaki_triton_amd as ozk
    xdt, sdt = [(torch.float64, torch.int8), (torch.float32, torch.float16),
                (torch.bfloat16, torch.int8)][(rows + K) % 3]
    g = torch.Generator().manual_seed(batch * 1000 + rows)
    X = torch.randn(batch, rows, K, generator=g, dtype=torch.float64).to(xdt)
    alpha = ozk.compute_split_bits(K, sdt, torch.int32 if sdt == torch.int8 else torch.float32)
    sl, sc = ozk.split_matrix(X.to(gpu), 2, alpha, sdt)
    torch.cuda.synchronize()
    osl, osc = oracle_split_batched(oracle, to_np(X), 2, alpha, sdt)
    assert_bitwise_equal(to_np(sc), osc, "scales")
    assert_bitwise_equal(to_np(sl), osl, "slices")


# both splits in one launch: whole rows beside columns of any pitch, in every class
# of K, and columns of A beside rows of B
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
@pytest.mark.parametrize("xdt,sdt", [(torch.float64, torch.int8), (torch.float32, torch.int8),
                                     (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("batch,M,N,K", [(3, 5, 7, 96), (4, 33, 111, 320), (3, 130, 63, 704),
                                         (2, 66, 97, 1344), (2, 34, 35, 2900), (1, 130, 111, 5600)])
def test_whole_rows_beside_any_columns(gpu, batch, M, N, K, xdt, sdt, ta, tb):
    import ozaki_triton_amd as ozk
    g = torch.Generator().manual_seed(M * N + K)
    A = torch.randn(batch, M, K, generator=g, dtype=torch.float64).to(xdt).to(gpu)
    B = torch.randn(batch, K, N, generator=g, dtype=torch.float64).to(xdt).to(gpu)
    A = A.mT.contiguous().mT if ta else A
    B = B.mT.contiguous().mT if tb else B
    got = ozk.ozaki_matmul(A, B, 3, sdt)
    # each operand split alone, from contiguous rows (checked against the oracle above)
    alpha = ozk.compute_split_bits(K, sdt, torch.int32 if sdt == torch.int8 else torch.float32)
    a_sl, a_sc = ozk.split_matrix(A.contiguous(), 3, alpha, sdt)
    b_sl, b_sc = ozk.split_matrix(B.mT.contiguous(), 3, alpha, sdt)
    want = ozk.cross_gemm(a_sl, b_sl.transpose(-1, -2), a_sc, b_sc, 3, xdt)
    torch.cuda.synchronize()
    assert_bitwise_equal(to_np(got), to_np(want), f"{ta} {tb}")


@pytest.mark.parametrize("batch,rows,K", [(1, (1 << 25) + 70, 516), (3, (1 << 22) - 1, 8)])
def test_more_rows_than_a_launch_counts(gpu, batch, rows, K):
    """Rows whose work-items are 2^32 and more (35 GB of input and slices), and
    batches cut between launches: the rows around the cuts as split alone."""
    import ozaki_triton_amd as ozk
    print(f"[rows] {batch}x{rows}x{K}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(K)
    X = torch.randint(-100, 101, (batch, rows, K), generator=g, dtype=torch.int8, device=gpu)
    sl, sc = ozk.split_matrix(X, 1, 7, torch.int8)
    for b in {0, batch - 1}:
        for at in {0, (1 << 23) - 2, (1 << 24) - 2, (1 << 25) - 2, rows - 4}:
            if at + 4 <= rows:
                wl, wc = ozk.split_matrix(X[b:b + 1, at:at + 4].contiguous(), 1, 7, torch.int8)
                torch.cuda.synchronize()
                assert torch.equal(sl[b:b + 1, :, at:at + 4], wl), (b, at)
                assert torch.equal(sc[b:b + 1, :, at:at + 4], wc), (b, at)
    del X, sl, sc
    torch.cuda.empty_cache()
