"""int8 slices with more bits than an int8 holds (alpha > 7, which split_matrix
takes from its caller): both ends clamped as in the oracle, the rest in the
residual."""
import pytest
import torch

from tests.helpers import assert_bitwise_equal, oracle_split_batched, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns", [False, True])
@pytest.mark.parametrize("xdt", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("alpha", [7, 8, 12])
def test_alpha_beyond_int8(oracle, gpu, alpha, xdt, columns):
    import ozaki_triton_amd as ozk
    g = torch.Generator().manual_seed(alpha)
    X = torch.randn(1, 24, 300, generator=g, dtype=torch.float64).to(xdt)
    Xd = X.to(gpu).mT.contiguous().mT if columns else X.to(gpu)
    sl, sc = ozk.split_matrix(Xd, 3, alpha, torch.int8)
    torch.cuda.synchronize()
    osl, osc = oracle_split_batched(oracle, to_np(X), 3, alpha, torch.int8)
    assert_bitwise_equal(to_np(sc), osc, "scales")
    assert_bitwise_equal(to_np(sl), osl, "slices")
