"""The matrix-core decoder weight gradient and its Adam step (clt_decoder_grad_tiles, clt_decoder_grad_adam_tiles) at the
edges of their tiles: 512 tokens, 16 features per group, 8 wavefronts x 4 groups per workgroup, 64 columns."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,T,F,d,per_token", [
    (1, 1, 4, 64, 2), (2, 512, 512, 64, 20), (2, 513, 513, 128, 40), (3, 37, 1030, 192, 1), (2, 1500, 40, 64, 30), (1, 300, 2000, 256, 900),
])
def test_grad_tiles_against_dense_products(L, T, F, d, per_token):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(T + F)
    act = torch.where(torch.rand(L, T, F, generator=g) < per_token / F, torch.randn(L, T, F, generator=g), torch.zeros(())).bfloat16()
    act[:, :, F // 2] = 0                                   # a feature that never fires
    flat = act.reshape(L * T, F)
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum((flat != 0).sum(1), 0)
    surv = engine.SurvivorList(row_ptr.to(dev), (flat != 0).nonzero()[:, 1].int().to(dev), flat[flat != 0].to(dev), T, F, L, torch.bfloat16)
    gm = torch.randn(L, T, d, generator=g).bfloat16()
    n_dec = L * (L + 1) // 2
    assert engine.grad_tiles_supported(T, d, F, L, surv.capacity, torch.bfloat16)
    ws = engine.Workspace(dev)
    lists = engine.feature_lists(surv, ws)
    ws.get("grad_tiles", nat.load().clt_grad_tiles_workspace_bytes(T, d, F, L, surv.capacity)).fill_(0xFF)      # must not matter
    got = engine.decoder_weight_grad(lists, surv, gm.to(dev), "none", ws=ws).cpu()
    assert torch.equal(got, engine.decoder_weight_grad(lists, surv, gm.to(dev), "none", ws=ws).cpu())
    slot = 0
    for s in range(L):
        for t in range(s, L):
            ref, mag = act[s].double().t() @ gm[t].double(), act[s].double().abs().t() @ gm[t].double().abs()
            n = (act[s] != 0).sum(0).double().unsqueeze(1)
            # exact products, one fp32 addition per token: each off by at most 2^-23 of what has been summed
            assert (got[slot].double() - ref).abs().le((n + 1) * 2.0 ** -23 * mag).all()
            slot += 1
    # the step: the row kernel is gradient-then-Adam bit for bit, and the two gradients agree to the bound above
    w = engine.alloc_packed(n_dec, F, d, torch.bfloat16, dev)
    w[:, :, :d] = (torch.rand(n_dec, F, d, generator=g) - 0.5).to(torch.bfloat16)
    m, v = 0.1 * torch.randn(n_dec, F, d, generator=g).to(dev), torch.rand(n_dec, F, d, generator=g).to(dev) + 0.1
    tiled = lambda x: x.view(n_dec, F, d // 64, 64).permute(0, 2, 1, 3).clone(memory_format=torch.contiguous_format)   # noqa: E731
    states = {"ref": (w.clone(), m.clone(), v.clone()), "rows": (w.clone(), m.clone(), v.clone()), "tiles": (w.clone(), tiled(m), tiled(v))}
    args = (1e-2, (0.9, 0.999), 1e-8, 3)
    engine.decoder_weight_grad_adam(lists, surv, gm.to(dev), *states["ref"], *args)
    for key in ("rows", "tiles"):
        engine.decoder_grad_adam_tiles(lists, surv, gm.to(dev), *states[key], *args, ws=ws)
    for i in (1, 2):
        back = states["tiles"][i].permute(0, 2, 1, 3).reshape(n_dec, F, d)
        assert torch.equal(back, states["rows"][i])
        assert torch.allclose(back, states["ref"][i], rtol=1e-5, atol=1e-5 * float(states["ref"][i].abs().max()))
    assert torch.equal(states["tiles"][0], states["rows"][0])
    step = (states["rows"][0].float() - states["ref"][0].float()).abs()
    # one bf16 ulp (weights below 0.5 in size and steps below 0.05: at most 2^-9) where a sum lies on a rounding boundary
    assert float(step.max()) <= 2.0 ** -8 and float((step > 0).float().mean()) < 1e-3
