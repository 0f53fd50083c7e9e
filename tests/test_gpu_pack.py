"""cross_gemm on slices the kernels cannot read in place (pack_kernel): rows that
are no whole 16-byte pieces, the [K, N] layout, other strides, a broadcast
operand; C bit for bit equal to that of the same slices in aligned,
zero-padded K-contiguous tensors."""
import pytest
import torch

from tests.helpers import assert_bitwise_equal, int_valued_slices, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sdt", [torch.int8, torch.float16, torch.float32])
@pytest.mark.parametrize("layout", ["rows", "columns", "strided"])
@pytest.mark.parametrize("batch,bcast", [(1, False), (3, False), (3, True)])
@pytest.mark.parametrize("M,N,K", [(5, 3, 1), (64, 64, 63), (65, 130, 67), (70, 129, 515)])
def test_packed_layouts(gpu, M, N, K, batch, bcast, layout, sdt):
    import ozaki_triton_amd as ozk
    L = 3
    g = torch.Generator().manual_seed(M + N + K)
    As, BsT, sa, sb = int_valued_slices(g, batch, L, M, N, K, sdt)
    if bcast:
        BsT, sb = BsT[:1], sb[:1]
    Kp = (K + 15) // 16 * 16

    def padded(x):
        y = torch.zeros(*x.shape[:-1], Kp, dtype=sdt)
        y[..., :K] = x
        return y.to(gpu)

    sa, sb = sa.to(gpu), sb.to(gpu)
    want = ozk.cross_gemm(padded(As), padded(BsT).transpose(-1, -2), sa, sb, L, torch.float64)
    Ad, Bd = As.to(gpu), BsT.to(gpu)
    if layout == "columns":     # A M-contiguous, B N-contiguous
        Ad = Ad.mT.contiguous().mT
        Bd = Bd.mT.contiguous().mT
    elif layout == "strided":   # every other element
        Ad = Ad.repeat_interleave(2, dim=-1)[..., ::2]
        Bd = Bd.repeat_interleave(2, dim=-1)[..., ::2]
    got = ozk.cross_gemm(Ad, Bd.transpose(-1, -2), sa, sb, L, torch.float64)
    torch.cuda.synchronize()
    assert_bitwise_equal(to_np(got), to_np(want), f"{layout} {sdt}")
