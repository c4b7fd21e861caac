"""Gradients of the kept activations where the lists end: every number of rows left over from a step, empty slices, and lists around
the 64 entries that a wavefront holds at once, against products in float64."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu

LENGTHS = list(range(19)) + [63, 64, 65, 70, 72]      # entries of a token in each of the eight feature slices


@pytest.mark.parametrize("d,dtype", [
    (512, torch.float32), (768, torch.float32), (1024, torch.float32), (2048, torch.float32),     # 2, 3, 4 and 8 pieces per lane
    (768, torch.bfloat16), (1536, torch.bfloat16), (2048, torch.bfloat16), (4096, torch.bfloat16),
])
def test_value_gradients_at_the_ends_of_lists(d, dtype):
    dev = torch.device("cuda:0")
    L, T, per_slice = 2, len(LENGTHS), 72
    F = 8 * per_slice
    g = torch.Generator().manual_seed(d)
    keep = torch.zeros(L, T, F, dtype=torch.bool)
    for s in range(L):
        for t in range(T):
            for sl in range(8):
                n = LENGTHS[(t + s * sl) % T]         # source 1: another length in every slice
                keep[s, t, sl * per_slice + torch.randperm(per_slice, generator=g)[:n]] = True
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(keep.view(L * T, F).sum(1), 0)
    col = keep.view(L * T, F).nonzero()[:, 1].int()
    surv = engine.SurvivorList(row_ptr.to(dev), col.to(dev), torch.ones(col.numel(), dtype=dtype, device=dev), T, F, L, dtype)
    w = torch.zeros(3, F, engine.decoder_pitch(d, dtype), dtype=dtype)
    w[:, :, :d] = torch.randn(3, F, d, generator=g).to(dtype)
    grad = torch.randn(L, T, d, generator=g)
    got = engine.decode_backward_values(surv, w.to(dev), grad.to(dev), "none").cpu().double()
    rows, gd = w[:, :, :d].double(), grad.double()
    dense = torch.stack([gd[0] @ rows[0].t() + gd[1] @ rows[1].t(), gd[1] @ rows[2].t()])
    size = torch.stack([gd[0].abs() @ rows[0].t().abs() + gd[1].abs() @ rows[1].t().abs(), gd[1].abs() @ rows[2].t().abs()])
    # a lane adds d / 64 products, six exchanges add the lanes, one addition the targets: so many roundings of 2^-24 per term
    assert bool(((got - dense[keep]).abs() <= size[keep] * (d / 64 + 8) * 2.0 ** -24).all())


@pytest.mark.parametrize("L,empty", [(1, ()), (2, (0,)), (5, (1, 2, 4)), (7, ()), (64, (0, 31, 32, 63)), (3, (0, 1))])
def test_value_gradients_of_sources_without_survivors(L, empty):
    dev = torch.device("cuda:0")
    T, F, d = 9, 24, 64
    g = torch.Generator().manual_seed(L)
    keep = torch.rand(L, T, F, generator=g) < 0.2
    for s in empty:
        keep[s] = False
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(keep.view(L * T, F).sum(1), 0)
    col = keep.view(L * T, F).nonzero()[:, 1].int()
    surv = engine.SurvivorList(row_ptr.to(dev), col.to(dev), torch.ones(col.numel(), device=dev), T, F, L, torch.float32)
    w = torch.zeros(L * (L + 1) // 2, F, engine.decoder_pitch(d, torch.float32))
    w[:, :, :d] = torch.randn(w.shape[0], F, d, generator=g)
    grad = torch.randn(L, T, d, generator=g)
    mask = (1 << L) - 1 if L < 5 else ((1 << L) - 1) & ~(1 << 3)         # (source 3 left out: its gradients are zeros)
    got = engine.decode_backward_values(surv, w.to(dev), grad.to(dev), "none", mask).cpu().double()
    rows, gd, dense, size = w[:, :, :d].double(), grad.double(), [], []
    for s in range(L):
        first = s * L - s * (s - 1) // 2
        on = float((mask >> s) & 1)
        dense.append(on * sum(gd[t] @ rows[first + t - s].t() for t in range(s, L)))
        size.append(sum(gd[t].abs() @ rows[first + t - s].t().abs() for t in range(s, L)))
    # d / 64 products per lane, six exchanges, one addition per target
    assert bool(((got - torch.stack(dense)[keep]).abs() <= torch.stack(size)[keep] * (d / 64 + 6 + L) * 2.0 ** -24).all())
