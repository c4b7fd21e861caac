"""k_encode_mfma over few stages of K and more tiles than workgroups: the shortest pipelines (one stage with the appended
one, two, three, four) and the turn from one tile to the next, with shifted tiles in both directions."""

import pytest
import torch

import crosslayer_coding_amd as cca

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("stages", [1, 2, 3, 4])
@pytest.mark.parametrize("with_bias", [True, False])
def test_products_over_few_stages(dtype, stages, with_bias):
    dev = torch.device("cuda")
    L, T, F, d = 3, 1030, 4364, stages * 128 // dtype.itemsize          # 5 x 18 tiles per layer, 256 workgroups
    gen = torch.Generator().manual_seed(stages)
    x = torch.randn(L, T, d, generator=gen).to(dtype).to(dev)
    w = (torch.randn(L, F, d, generator=gen) * d ** -0.5).to(dtype).to(dev)
    b = torch.randn(L, F, generator=gen).to(dtype).to(dev) if with_bias else None
    for _ in range(2):
        out = torch.full((L, T, F), float("nan"), dtype=dtype, device=dev)
        cca.engine.encode(x, w, b, out)
        for l in range(L):
            ref = x[l].double() @ w[l].double().T + (b[l].double() if with_bias else 0.0)
            mag = x[l].double().abs() @ w[l].double().abs().T + (b[l].double().abs() if with_bias else 0.0)
            # one rounding of the result plus fp32 sums of d products in any order
            bound = torch.finfo(dtype).eps / 2 * ref.abs() + (d + 8) * 2.0 ** -24 * mag + (2.0 ** -24 if dtype == torch.float16 else 0.0)
            err = (out[l].double() - ref).abs()
            assert bool((err <= bound).all()), (l, float((err - bound).max()))
