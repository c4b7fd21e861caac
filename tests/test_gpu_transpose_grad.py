"""A decoder's gradient in its parameter's layout and dtype (clt_transpose_grad) is torch's cast and transpose bit for bit, at
whole and ragged 64 x 64 tiles."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("F,d", [(8, 4), (64, 64), (72, 68), (1000, 100), (136, 768), (4104, 36), (30, 64), (64, 30)])
def test_parameter_gradient(F, d, dtype):
    g = torch.randn(F, d, device="cuda")
    g[0, 0], g[-1, -1], g[F // 2, 0], g[0, d // 2] = float("inf"), float("nan"), -float("inf"), 3.39e38
    got, want = engine.parameter_gradient(g.t(), dtype), g.t().to(dtype)
    assert got.dtype == dtype and got.shape == (d, F)
    if F % 8 == 0 and d % 4 == 0:
        assert got.is_contiguous()
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan) and torch.equal(got.masked_fill(nan, 0), want.masked_fill(nan, 0))
    assert torch.equal(engine.parameter_gradient(g, dtype).isnan(), nan.t())      # already in its layout
