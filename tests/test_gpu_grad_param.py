"""Decoder gradients in the parameters' layout (clt_decoder_grad_param_tiles) are the fp32 rows of clt_decoder_grad_tiles rounded and
transposed, bit for bit, at the edges of a workgroup's 512 features, non-finite sums included."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,T,F,d,per_token", [
    (1, 2, 8, 64, 6), (2, 513, 512, 64, 20), (2, 300, 520, 128, 40), (3, 37, 1032, 192, 3), (2, 1500, 2040, 64, 30), (2, 64, 4104, 64, 9),
])
def test_parameter_layout(L, T, F, d, per_token):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(T + F)
    act = torch.where(torch.rand(L, T, F, generator=g) < per_token / F, torch.randn(L, T, F, generator=g), torch.zeros(())).bfloat16()
    flat = act.reshape(L * T, F)
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum((flat != 0).sum(1), 0)
    surv = engine.SurvivorList(row_ptr.to(dev), (flat != 0).nonzero()[:, 1].int().to(dev), flat[flat != 0].to(dev), T, F, L, torch.bfloat16)
    gm = torch.randn(L, T, d, generator=g).bfloat16()
    gm[-1, T // 2, 3], gm[0, 0, d - 1] = float("inf"), float("nan")
    gm = gm.to(dev)
    lists = engine.feature_lists(surv)
    rows = engine.decoder_weight_grad(lists, surv, gm, "none")
    got = engine.decoder_parameter_grad(lists, surv, gm)
    assert got.shape == (L * (L + 1) // 2, d, F) and got.dtype == torch.bfloat16 and got.is_contiguous()
    want = rows.transpose(1, 2).to(torch.bfloat16)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0)) and torch.equal(got.isinf(), want.isinf())


def test_other_widths_are_left_to_the_rows():
    dev = torch.device("cuda:0")
    L, T, F, d = 1, 20, 36, 64
    surv = engine.SurvivorList(torch.arange(T + 1, dtype=torch.int32, device=dev), torch.zeros(T, dtype=torch.int32, device=dev),
                               torch.ones(T, device=dev).bfloat16(), T, F, L, torch.bfloat16)
    gm = torch.ones(L, T, d, device=dev).bfloat16()
    lists = engine.feature_lists(surv)
    assert engine.decoder_parameter_grad(lists, surv, gm) is None           # F no multiple of 8
    assert engine.decoder_parameter_grad(lists, surv, gm[:, :, :40].contiguous()) is None


@pytest.mark.parametrize("L,T,F,d,per_token", [(2, 300, 520, 128, 40), (23, 5, 16, 64, 2)])
def test_addresses_of_their_own(L, T, F, d, per_token):
    # (276 decoders: the addresses go to the device in two launches)
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(T + F)
    act = torch.where(torch.rand(L, T, F, generator=g) < per_token / F, torch.randn(L, T, F, generator=g), torch.zeros(())).bfloat16()
    flat = act.reshape(L * T, F)
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum((flat != 0).sum(1), 0)
    surv = engine.SurvivorList(row_ptr.to(dev), (flat != 0).nonzero()[:, 1].int().to(dev), flat[flat != 0].to(dev), T, F, L, torch.bfloat16)
    gm = torch.randn(L, T, d, generator=g).bfloat16().to(dev)
    lists = engine.feature_lists(surv)
    together, apart = engine.decoder_parameter_grad(lists, surv, gm), engine.decoder_parameter_grad(lists, surv, gm, separate=True)
    assert len(apart) == L * (L + 1) // 2 and all(torch.equal(a, b) for a, b in zip(together, apart))


@pytest.mark.parametrize("tying", ["none", "per_source", "per_target"])
def test_gradients_share_no_memory(tying):
    import crosslayer_coding_amd as cca
    from crosslayer_coding_amd import synth
    dev = torch.device("cuda:0")
    wl = synth.Workload("apart", 4, 3, 64, 512, 200, "bfloat16", k=10, decoder_tying=tying)
    model, x, _ = synth.build_model(wl, dev, 1)
    recs = model({l: x[l] for l in range(3)})
    sum((r.float() ** 2).mean() for r in recs.values()).backward()
    grads = [(n, p.grad) for n, p in model.named_parameters() if p.grad is not None]
    assert len(grads) >= 9
    for name, grad in grads:
        assert grad.dtype == torch.bfloat16 and grad.untyped_storage().nbytes() == 2 * grad.numel(), name
    assert cca is not None
