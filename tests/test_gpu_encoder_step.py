"""The encoder weights' Adam step inside the weight-gradient kernel against gradient-then-Adam, bit for bit: every number of pieces a
lane holds, rows that are no whole number of pieces per wavefront, features without entries and with more than a wavefront holds."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat
from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dtype", [
    (8, torch.bfloat16), (136, torch.bfloat16), (768, torch.bfloat16), (1024, torch.bfloat16), (1032, torch.bfloat16), (2048, torch.bfloat16), (256, torch.bfloat16), (1280, torch.bfloat16), (1792, torch.bfloat16),
    (4, torch.float32), (68, torch.float32), (512, torch.float32), (768, torch.float32), (1024, torch.float32),
])
def test_encoder_step_in_the_gradient_kernel(d, dtype):
    dev = torch.device("cuda:0")
    L, F, T = 3, 37, 211
    g = torch.Generator().manual_seed(d)
    counts = torch.randint(0, 12, (L, F), generator=g)
    counts[0, :3], counts[1, 5], counts[2, F - 1] = 0, 150, 65
    ptr = torch.zeros(L * F + 1, dtype=torch.int32)
    ptr[1:] = torch.cumsum(counts.view(-1), 0)
    n = int(ptr[-1])
    lists = tuple(t.to(dev) for t in (ptr, torch.randint(0, T, (n,), generator=g).int(), torch.randperm(n, generator=g).int()))
    dval = torch.randn(n, generator=g).to(dev)
    x = torch.randn(L, T, d, generator=g).to(dtype).to(dev)
    w = torch.randn(L, F, d, generator=g).to(dtype).to(dev)
    m, v = torch.randn(L, F, d, generator=g).to(dev), torch.rand(L, F, d, generator=g).to(dev)
    w2, m2, v2 = w.clone(), m.clone(), v.clone()
    dw, db = engine.encoder_weight_grad(lists, dval, x, F)
    nat.check(nat.load().clt_adam_step(nat.ptr(w2), nat.ptr(dw), nat.ptr(m2), nat.ptr(v2), w2.numel(), 1e-2, 0.9, 0.999, 1e-8, 4,
                                       nat.dtype_code(dtype), nat.current_stream(dev)), "clt_adam_step")
    assert engine.encoder_step_fits(d, dtype)
    got = engine.encoder_weight_grad_adam(lists, dval, x, w, m, v, 1e-2, (0.9, 0.999), 1e-8, 4)
    assert torch.equal(got, db) and torch.equal(w, w2) and torch.equal(m, m2) and torch.equal(v, v2)


def test_wide_rows_keep_the_two_calls():
    assert not engine.encoder_step_fits(2056, torch.bfloat16) and not engine.encoder_step_fits(1028, torch.float32)
    assert not engine.encoder_step_fits(768, torch.float16)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_a_step_that_finds_no_memory_leaves_the_model_as_it_was(monkeypatch, dtype):
    """The workspace of the decoder step is what a longer batch outgrows first: the call raises before anything has moved, and the
    same call afterwards is the first step of a model that never raised."""
    import crosslayer_coding_amd as cca
    from crosslayer_coding_amd import synth
    dev = torch.device("cuda:0")
    wl = synth.Workload("retry", 3, 3, 128, 512, 300, dtype, k=12)
    ends = []
    for fails in (False, True):
        model, x, _ = synth.build_model(wl, dev, 1)
        y = synth.make_targets(wl, dev, 1)
        opt, inputs, targets = cca.CLTAdam(model, lr=1e-2), {l: x[l] for l in range(3)}, {l: y[l] for l in range(3)}

        def state():
            return [t.clone() for t in (*model.encoder_module.stacked(), model.decoder_module.packed(), *opt.decoder_moments(),
                                        *opt.state["enc_w"], *opt.state["enc_b"], *opt.state["dec_b"])]

        if fails:
            before, get = state(), engine.Workspace.get
            with monkeypatch.context() as patch:
                def no_room(self, name, nbytes):
                    if name in ("grad_tiles", "decoder_tiles"):
                        raise torch.OutOfMemoryError(name)
                    return get(self, name, nbytes)
                patch.setattr(engine.Workspace, "get", no_room)
                with pytest.raises(torch.OutOfMemoryError):
                    model.training_step(inputs, targets, opt)
            assert opt.step_count == 0 and all(torch.equal(a, b) for a, b in zip(before, state()))
        loss = model.training_step(inputs, targets, opt)
        ends.append([loss] + state())
    assert all(torch.equal(a, b) for a, b in zip(*ends))


@pytest.mark.parametrize("T,taken", [(256, True), (700, False)])
def test_a_training_step_takes_it_for_short_lists(monkeypatch, T, taken):
    """24 of 128 features fire per token: lists of 48 and of 131 entries; the same bits either way."""
    import crosslayer_coding_amd as cca
    from crosslayer_coding_amd import synth
    wl, ends, ran = synth.Workload("lists", 5, 2, 64, 128, T, "bfloat16", k=24), [], []
    real = engine.encoder_weight_grad_adam
    monkeypatch.setattr(engine, "encoder_weight_grad_adam", lambda *a: ran.append(1) or real(*a))
    for fuse in (True, False):
        model, x, _ = synth.build_model(wl, torch.device("cuda:0"), 1)
        y = synth.make_targets(wl, torch.device("cuda:0"), 1)
        opt = cca.CLTAdam(model, lr=1e-2)
        opt.fuse_encoder_step = fuse
        model.training_step({l: x[l] for l in range(2)}, {l: y[l] for l in range(2)}, opt)
        ends.append([t.clone() for t in (*model.encoder_module.stacked(), *opt.state["enc_w"], *opt.state["enc_b"])])
    assert ran == ([1] if taken else [])
    assert all(torch.equal(a, b) for a, b in zip(*ends))
