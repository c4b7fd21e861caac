"""The sampled cut of the batch-wide selection where its sample changes size: 16384 keys down to one element in 512 kept,
65536 down to one in 2048, 262144 below, and a problem that is smaller than its sample.  The survivors are exact whatever
the sample says, so they are compared one for one with a stable sort."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L,T,F,k", [
    (1, 300, 1024, 2), (1, 300, 1024, 1), (2, 150, 2048, 1), (1, 200, 2056, 1), (3, 90, 4096, 2), (1, 63, 4097, 1), (2, 1, 8192, 1),
    (1, 64, 4096, 1),
])
@pytest.mark.parametrize("global_mode", [False, True])
def test_sampled_cut_keeps_the_selection_exact(L, T, F, k, global_mode, dtype):
    g = torch.Generator().manual_seed(T * 3 + F)
    pre = torch.randn(L, T, F, generator=g).to(dtype)
    dev = torch.device("cuda:0")
    x = pre.to(dev)
    stats = engine.colstats(x) if global_mode else None
    surv = engine.batchtopk_select(x, k, global_mode, stats=stats)
    got = torch.zeros(L * T, F, dtype=torch.bool)
    rows = torch.repeat_interleave(torch.arange(L * T), torch.diff(surv.row_ptr.cpu().long()))
    n = int(surv.row_ptr[-1])
    got[rows, surv.col[:n].cpu().long()] = True
    if global_mode:
        mean, denom = (s.cpu() for s in stats)
        rank = torch.stack([((pre[l].float() - mean[l]).to(dtype).float() / denom[l]).to(dtype).float() for l in range(L)])
        flat = rank.permute(1, 0, 2).reshape(1, -1)                       # token-major: all layers of a token in turn
    else:
        flat = pre.float().reshape(L, -1)
    want = torch.zeros_like(flat, dtype=torch.bool)
    want.scatter_(1, torch.sort(flat, dim=1, descending=True, stable=True).indices[:, :k * T], True)
    want = want.view(T, L, F).permute(1, 0, 2) if global_mode else want.view(L, T, F)
    assert n == want.sum() and torch.equal(got.view(L, T, F), want)
