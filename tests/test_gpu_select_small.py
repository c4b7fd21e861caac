"""Per-layer BatchTopK of small problems (k_select_small) against a stable sort: sizes around its limits, ties, negative
thresholds, NaNs and infinities, rows that keep nothing or everything."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L,T,F,k", [
    (1, 1, 1, 1), (2, 3, 5, 2), (3, 32, 1024, 16), (1, 2048, 16, 3), (2, 2047, 9, 1), (1, 2049, 8, 2), (1, 32, 1023, 1023), (2, 7, 100, 99),
    (1, 1, 32768, 200), (1, 16, 4096, 5), (1, 8, 4097, 60), (2, 1030, 20, 30),
])
@pytest.mark.parametrize("kind", ["normal", "ties", "special"])
def test_small_selection_is_exact(L, T, F, k, kind, dtype):
    g = torch.Generator().manual_seed(T * 7 + F)
    pre = torch.randn(L, T, F, generator=g)
    if kind == "ties":
        pre = torch.randint(-2, 2, (L, T, F), generator=g).float() * 0.5          # four values, -0.0 and 0.0 among them
        pre[0, 0, 0] = -0.0
    if kind == "special":
        at = torch.rand(L, T, F, generator=g)
        pre[at < 0.02] = float("nan")
        pre[at > 0.97] = float("inf")
        pre[(at > 0.5) & (at < 0.55)] = -float("inf")
    x = pre.to(dtype)
    surv = engine.batchtopk_select(x.cuda(), k, False)
    n = L * min(k * T, T * F)
    assert int(surv.row_ptr[-1]) == n and surv.col.numel() == n
    rows = torch.repeat_interleave(torch.arange(L * T), torch.diff(surv.row_ptr.cpu().long()))
    col = surv.col.cpu().long()
    rank = x.float().masked_fill(x.isnan(), float("inf")).reshape(L, -1).double()
    rank[x.reshape(L, -1).isnan()] = 1e300                                          # a NaN ranks above everything
    rank[rank == float("inf")] = 1e299
    idx = torch.sort(rank, dim=1, descending=True, stable=True).indices[:, :n // L]
    want = torch.zeros(L, T * F, dtype=torch.bool).scatter_(1, idx, True).view(L * T, F)
    got = torch.zeros(L * T, F, dtype=torch.bool)
    got[rows, col] = True
    assert torch.equal(got, want)
    same = (rows[1:] > rows[:-1]) | (col[1:] > col[:-1])
    assert bool(same.all())                                                         # ascending within a row
    v = x.reshape(L * T, F)[rows, col]
    got_v = surv.val.cpu()
    assert torch.equal(got_v.isnan(), v.isnan()) and torch.equal(got_v[~v.isnan()], v[~v.isnan()])
