"""The gather decode of short batches in one launch over all (source, target) pairs gives the bits of a launch per source:
the same rows, alone and as the first rows of a batch that is too long for one launch."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,d,F,dtype,tying,route", [
    (12, 768, 600, torch.bfloat16, "none", nat.ROUTE_QUARTER), (12, 768, 520, torch.float32, "none", nat.ROUTE_QUARTER),
    (12, 1024, 640, torch.float16, "per_source", nat.ROUTE_QUARTER), (14, 640, 528, torch.bfloat16, "none", nat.ROUTE_LINE),
    (13, 672, 512, torch.float32, "none", nat.ROUTE_LINE),
])
@pytest.mark.parametrize("T,span,mask", [(1, None, None), (37, None, None), (9, (3, 8), 0b1010110101), (5, (2, 4), 0)])
def test_one_launch_and_many(monkeypatch, L, d, F, dtype, tying, route, T, span, mask):
    monkeypatch.setattr(engine, "SLICED_DECODE_MIN_ROWS", 0)
    for route_price in ("clt_decode_tiles_wanted", "clt_decode_rows_wanted"):      # the gathers only
        monkeypatch.setattr(nat.load(), route_price, lambda *a: 0, raising=False)
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(T + d)
    long = (256 << 20) // (L * (L + 1) * d * 4) + 8
    assert engine.decode_route(T, d, F, L, tying, dtype, rows=1 << 20) == route
    n_dec = L * (L + 1) // 2 if tying == "none" else L
    w = engine.alloc_packed(n_dec, F, d, dtype, dev)
    w[:, :, :d] = torch.randn(n_dec, F, d, generator=g).to(dtype).to(dev)
    keep = torch.rand(L, T, F, generator=g) < 0.15
    keep[:, 0, :70] = True                                  # more than 64 of a slice
    keep[1] = False                                         # a source without survivors
    vals = torch.randn(L, T, F, generator=g).to(dtype)
    bias, outs = torch.randn(L, d, generator=g).to(dev), []
    a, b = span or (0, L)
    for rows in (T, long):
        full = torch.zeros(L, rows, F, dtype=torch.bool)
        full[:, :T] = keep
        ptr = torch.zeros(L * rows + 1, dtype=torch.int32)
        ptr[1:] = torch.cumsum(full.view(L * rows, F).sum(1), 0)
        surv = engine.SurvivorList(ptr.to(dev), full.view(L * rows, F).nonzero()[:, 1].int().to(dev), vals[keep].to(dev), rows, F, L, dtype)
        outs.append(engine.decode_sparse(surv, w, tying, d, bias_sum=bias, t_begin=a, t_end=b, src_mask=mask,
                                         ws=engine.Workspace(dev), out_f32=True)[a:b, :T].clone())
    assert torch.equal(outs[0], outs[1])
    act = torch.where(keep, vals, torch.zeros((), dtype=dtype)).double()
    for t in range(a, b):
        ref, mag = bias[t].cpu().double().expand(T, d).clone(), bias[t].cpu().double().abs().expand(T, d).clone()
        for s in range(t + 1):
            if mask is None or (mask >> s) & 1:
                m = w[s if tying != "none" else s * L - s * (s - 1) // 2 + t - s, :, :d].cpu().double()
                ref += act[s] @ m
                mag += act[s].abs() @ m.abs()
        n = 2.0 + float(keep.sum(2).sum(0).max())
        # exact products; at most n additions in fp32, each off by 2^-24 of what has been summed
        assert bool(((outs[0][t - a].cpu().double() - ref).abs() <= n * 2.0 ** -24 * mag).all())
