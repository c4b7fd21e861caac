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
