"""Selections whose sampled cut fails in some of the layers: those layers go through the pass again, by more workgroups, which share
the parts of the candidate pool that the first pass left."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def _sampled(n):
    """Where the selection takes its sample of a layer of n elements (hash_index), for more samples than it takes."""
    out = []
    for i in range(65536):
        x = ((i + 1) * 0x9E3779B97F4A7C15) & M64
        x ^= x >> 29
        x = (x * 0xBF58476D1CE4E5B9) & M64
        x ^= x >> 32
        out.append((x * n) >> 64)
    return torch.tensor(out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("L,T,F,k,bad", [
    (64, 300, 1032, 240, [5]),         # 16 workgroups a layer in the first pass, 38 in the second; more kept than sampled
    (64, 300, 1032, 240, [0, 17, 63]),
    (3, 300, 1032, 240, [1]),          # the same number in both
    (40, 29, 8192, 2600, [7]),         # rows cut into parts; a third of all elements kept
])
def test_layers_whose_cut_failed_are_selected_again(L, T, F, k, bad, dtype):
    dev, g = torch.device("cuda:0"), torch.Generator().manual_seed(L + T)
    pre = torch.randn(L, T, F, generator=g).to(dtype).to(dev)
    at = _sampled(T * F).to(dev)
    for l in bad:                      # nothing but the sample reaches what the sample says is the cut
        pre.view(L, -1)[l][at] += 16.0
    surv = engine.batchtopk_select(pre, k, False)
    flat = pre.view(L, -1)
    want = torch.zeros_like(flat, dtype=torch.bool)
    want.scatter_(1, torch.sort(flat, dim=1, descending=True, stable=True).indices[:, :k * T], True)
    want = want.view(L * T, F)
    n = int(surv.row_ptr[-1])
    assert n == int(want.sum()) and torch.equal(torch.diff(surv.row_ptr.long()), want.sum(1))
    rows, cols = want.nonzero(as_tuple=True)
    assert torch.equal(surv.col[:n].long(), cols) and torch.equal(surv.val[:n], pre.view(L * T, F)[rows, cols])


@pytest.mark.parametrize("bad", [[2], [0, 11]])
def test_layers_whose_collected_candidates_overflowed_are_selected_again(bad):
    dev, g = torch.device("cuda:0"), torch.Generator().manual_seed(1)
    L, T, F, d, k = 12, 700, 1536, 64, 9
    x = torch.randint(-1, 2, (L, T, d), generator=g).float()
    w = torch.randint(-1, 2, (L, F, d), generator=g).float()
    b = torch.randint(-2, 3, (L, F), generator=g).float()
    for l in bad:                      # every element is at the cut: more candidates than the pool holds
        w[l], b[l] = 0.0, 1.0
    x, w, b = (t.to(dev, torch.bfloat16) for t in (x, w, b))
    pre, ws = engine.encode(x, w, b), engine.Workspace(dev)
    got = engine.collect_select(engine.encode_collect(x, w, b, k, torch.empty_like(pre), ws))
    flat = pre.view(L, -1).float()
    want = torch.zeros_like(flat, dtype=torch.bool)
    want.scatter_(1, torch.sort(flat, dim=1, descending=True, stable=True).indices[:, :k * T], True)
    want = want.view(L * T, F)
    n = int(got.row_ptr[-1])
    assert n == int(want.sum()) and torch.equal(torch.diff(got.row_ptr.long()), want.sum(1))
    assert torch.equal(got.col[:n].long(), want.nonzero()[:, 1])
