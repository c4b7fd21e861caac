"""The float32 decode from LDS tiles (clt_decode_rows) against dense products in float64, at the edges of its tiles: 512
features, 16 tokens per wavefront, 16 wavefronts per workgroup, 8 entries per record, 4 records per slot, 32 columns."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,T,F,d,per_token,tying,heavy,span,mask", [
    (1, 1, 8, 32, 3, "none", False, None, None),                 # less than one of everything
    (2, 16, 512, 64, 32, "none", False, None, None),             # exactly one group, one tile
    (3, 17, 513, 96, 60, "none", False, None, None),             # one token and one feature over
    (3, 15, 1024, 32, 200, "per_source", True, None, None),      # runs of 512 entries
    (2, 257, 1300, 160, 20, "none", False, None, None),          # a workgroup's tokens and one more
    (4, 300, 4096, 64, 1, "none", True, None, None),             # most runs empty
    (2, 530, 640, 256, 40, "per_source", False, None, None),
    (5, 40, 1100, 64, 30, "none", False, (1, 4), 0b10110),       # some targets, some sources
    (3, 20, 600, 32, 30, "none", False, None, 0),                # no source at all
])
def test_decode_rows_against_dense_products(L, T, F, d, per_token, tying, heavy, span, mask):
    dev, lib = torch.device("cuda:0"), nat.load()
    g = torch.Generator().manual_seed(T + F)
    keep = torch.rand(L, T, F, generator=g) < per_token / F
    if heavy:                                               # one token with every feature, one source with next to none
        keep[:, T // 2] = True
        keep[1, :, F // 2:] = False
    act = torch.where(keep, torch.randn(L, T, F, generator=g), torch.zeros(()))
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(keep.view(L * T, F).sum(1), 0)
    n = int(row_ptr[-1])
    a, b = span or (0, L)
    mask = (1 << L) - 1 if mask is None else mask
    n_dec = L if tying == "per_source" else L * (L + 1) // 2
    w = engine.alloc_packed(n_dec, F, d, torch.float32, dev)
    w[:, :, :d] = torch.randn(n_dec, F, d, generator=g).to(dev)
    bias, skip = torch.randn(L, d, generator=g), torch.randn(L, T, d, generator=g)
    col, val = keep.view(L * T, F).nonzero()[:, 1].int().to(dev), act[keep].to(dev)
    ptr_d, bias_d, skip_d = row_ptr.to(dev), bias.to(dev), skip.to(dev)
    ws = torch.full((lib.clt_decode_rows_workspace_bytes(T, d, F, L, n),), 0xFF, dtype=torch.uint8, device=dev)
    outs = []
    for k in range(2):                                      # the second pass meets a workspace in use
        out = torch.full((L, T, d), 7.0, device=dev)
        nat.check(lib.clt_decode_rows(nat.ptr(ptr_d), nat.ptr(col), nat.ptr(val), nat.ptr(w), nat.ptr(bias_d), nat.ptr(skip_d),
                                      nat.ptr(out), T, d, F, L, nat.TYING[tying], a, b, mask, n, nat.ptr(ws), ws.numel(),
                                      nat.current_stream(dev)), "clt_decode_rows")
        outs.append(out.cpu())
    assert torch.equal(*outs)
    got, wc = outs[0], w.cpu()[:, :, :d].double()
    for t in range(L):
        if not a <= t < b:
            assert bool((got[t] == 7.0).all())              # not asked for
            continue
        ref, mag = bias[t].double() + skip[t].double(), bias[t].double().abs() + skip[t].double().abs()
        n_t = 0
        for s in range(t + 1):
            if (mask >> s) & 1:
                m = wc[s if tying == "per_source" else s * L - s * (s - 1) // 2 + t - s]
                ref, mag = ref + act[s].double() @ m, mag + act[s].double().abs() @ m.abs()
                n_t = n_t + keep[s].sum(1, keepdim=True)
        # one rounding per multiply-add or addition, each at most 2^-24 of what has been summed
        assert bool(((got[t].double() - ref).abs() <= (n_t + 8.0) * 2.0 ** -24 * mag).all())


def test_decode_rows_is_chosen_and_agrees_with_the_gather(monkeypatch):
    dev, lib = torch.device("cuda:0"), nat.load()
    L, T, F, d, k = 8, 1024, 3072, 768, 150
    assert lib.clt_decode_rows_wanted(T, d, F, L, L, L * T * k, nat.TYING["none"], nat.CLT_F32) == 1
    assert lib.clt_decode_rows_wanted(T, d, F, L, L, L * T * k, nat.TYING["per_target"], nat.CLT_F32) == 0
    assert lib.clt_decode_rows_wanted(T, d + 8, F, L, L, L * T * k, nat.TYING["none"], nat.CLT_F32) == 0
    assert lib.clt_decode_rows_wanted(2, d, F, L, L, L * 2 * k, nat.TYING["none"], nat.CLT_F32) == 0
    g = torch.Generator().manual_seed(3)
    pre = torch.randn(L, T, F, generator=g).to(dev)
    surv = engine.batchtopk_select(pre, k, False)
    w = engine.alloc_packed(L * (L + 1) // 2, F, d, torch.float32, dev)
    w[:, :, :d] = torch.randn(L * (L + 1) // 2, F, d, generator=g).to(dev)
    ws = engine.Workspace(dev)
    got = engine.decode_sparse(surv, w, "none", d, ws=ws)
    assert "decode_rows" in ws._bufs
    monkeypatch.setattr(lib, "clt_decode_rows_wanted", lambda *a: 0)
    ref = engine.decode_sparse(surv, w, "none", d, ws=ws)
    assert float((got - ref).norm() / ref.norm()) < 1e-6
