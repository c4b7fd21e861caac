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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L,T,F,k", [
    (2, 5, 16384, 30),             # rows cut into 16 parts
    (3, 40, 6144, 7),              # into 4, the last step of a part half empty
    (1, 77, 24584, 200),           # 8 * 3073 columns: not cut
    (2, 1300, 2056, 3),            # 2600 rows, too short to cut
    (12, 700, 2048, 1),            # enough rows
])
@pytest.mark.parametrize("kind", ["ties", "special"])
@pytest.mark.parametrize("global_mode", [False, True])
def test_selection_of_cut_rows_is_exact(L, T, F, k, kind, global_mode, dtype):
    g = torch.Generator().manual_seed(T * 5 + F)
    if kind == "ties":
        pre = torch.randint(-3, 3, (L, T, F), generator=g).float() * 0.5             # -0.0 and 0.0 among them
        pre[:, ::2][pre[:, ::2] == 0] = -0.0
    else:
        pre = torch.randn(L, T, F, generator=g)
        at = torch.rand(L, T, F, generator=g)
        pre[at < 0.002] = float("nan")
        pre[at > 0.999] = float("inf")
        pre[(at > 0.5) & (at < 0.52)] = -float("inf")
    pre = pre.to(dtype)
    if kind == "special":          # NaNs of the other sign too
        view = pre.view(torch.int32 if dtype == torch.float32 else torch.int16)
        view[:, 1::3] = torch.where(pre[:, 1::3].isnan(), view[:, 1::3] | torch.iinfo(view.dtype).min, view[:, 1::3])
    dev = torch.device("cuda:0")
    if global_mode:                # statistics of ordinary numbers, negative bounds among them
        mean = torch.randn(L, F, generator=g).to(dtype).float()
        denom = (torch.rand(L, F, generator=g) + 0.5).to(dtype).float()
        stats = (mean.to(dev), denom.to(dev))
        rank = torch.stack([((pre[l].float() - mean[l]).to(dtype).float() / denom[l]).to(dtype).float() for l in range(L)])
        rank = rank.permute(1, 0, 2).reshape(1, -1).double()
    else:
        stats, rank = None, pre.float().reshape(L, -1).double()
    surv = engine.batchtopk_select(pre.to(dev), k, global_mode, stats=stats)
    rank = torch.where(rank.isnan(), 1e300, torch.where(rank == float("inf"), 1e299, rank))
    want = torch.zeros_like(rank, dtype=torch.bool)
    want.scatter_(1, torch.sort(rank, dim=1, descending=True, stable=True).indices[:, :k * T], True)
    want = (want.view(T, L, F).permute(1, 0, 2) if global_mode else want.view(L, T, F)).reshape(L * T, F)
    n = int(surv.row_ptr[-1])
    counts = torch.diff(surv.row_ptr.cpu().long())
    assert n == want.sum() and torch.equal(counts, want.sum(1))
    rows, cols = want.nonzero(as_tuple=True)
    assert torch.equal(surv.col[:n].cpu().long(), cols)
    got, ref = surv.val[:n].cpu(), pre.reshape(L * T, F)[rows, cols]
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[~got.isnan()], ref[~ref.isnan()])
