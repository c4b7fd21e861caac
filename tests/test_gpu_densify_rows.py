"""Dense activations from survivor lists row by row (k_densify_rows) against an index assignment."""

import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,out_f32", [(torch.float32, False), (torch.bfloat16, False), (torch.bfloat16, True),
                                           (torch.float16, False), (torch.float16, True)])
@pytest.mark.parametrize("L,T,F", [(1, 1, 8), (2, 5, 13), (2, 7, 1024), (1, 3, 8200), (1, 5, 16384), (2, 3, 40008)])
def test_densify(L, T, F, dtype, out_f32):
    torch.manual_seed(F)
    dense = torch.randn(L, T, F, device="cuda").to(dtype)
    keep = torch.rand(L, T, F, device="cuda") < 0.1
    keep[0, 0] = True                        # a full row ..
    keep[-1, -1, :] = False                  # .. and an empty one
    if T > 2:
        keep[0, 2, 0] = keep[0, 2, F - 1] = True
    rows = keep.view(L * T, F)
    ptr = torch.zeros(L * T + 1, dtype=torch.int32, device="cuda")
    ptr[1:] = rows.sum(1).cumsum(0).to(torch.int32)
    col = rows.nonzero()[:, 1].to(torch.int32)
    surv = engine.SurvivorList(ptr, col, dense[keep], T, F, L, dtype)
    got = engine.densify(surv, out_f32=out_f32)
    want = torch.where(keep, dense, torch.zeros_like(dense))
    assert torch.equal(got, want.float() if out_f32 else want)
