"""Float32 decoder gradients from LDS tiles with the Adam step in place, at the edges of tiles, groups and records, against float64 gradients
and the general kernel."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


def _problem(L, T, F, d, density, seed, crowded=False):
    g = torch.Generator().manual_seed(seed)
    keep = torch.rand(L, T, F, generator=g) < density
    if crowded:                                            # features that fire on every token: records by the hundred
        keep[:, :, : min(16, F)] = True
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(keep.view(L * T, F).sum(1), 0)
    col = keep.view(L * T, F).nonzero()[:, 1].int()
    dense = torch.where(keep, torch.randn(L, T, F, generator=g), torch.zeros(()))
    surv = engine.SurvivorList(row_ptr.cuda(), col.cuda(), dense[keep].cuda(), T, F, L, torch.float32)
    n_dec = L * (L + 1) // 2
    w = torch.zeros(n_dec, F, engine.decoder_pitch(d, torch.float32))
    w[:, :, :d] = torch.randn(n_dec, F, d, generator=g)
    m, v = torch.zeros(n_dec, F, d), torch.zeros(n_dec, F, d)
    return surv, dense, w.cuda(), m.cuda(), v.cuda(), torch.randn(L, T, d, generator=g)


@pytest.mark.parametrize("L,T,F,d,density,crowded,by_tile", [
    (1, 1, 3, 32, 0.7, False, False),              # one token, less than a group
    (2, 511, 129, 64, 0.05, False, True),          # one feature past a workgroup, a token short of a tile
    (3, 513, 300, 96, 0.03, False, False),         # a token past a tile
    (2, 1300, 250, 160, 0.02, True, True),         # three tiles, full records in plenty
    (4, 700, 1031, 32, 0.002, False, False),       # most runs of one entry or none
])
def test_step_from_tiles(L, T, F, d, density, crowded, by_tile):
    surv, dense, w, m, v, g = _problem(L, T, F, d, density, T + F, crowded)
    lists, gd = engine.feature_lists(surv), g.cuda()
    tile = (lambda a: a.view(-1, F, d // 8, 8).permute(0, 2, 1, 3).contiguous()) if by_tile else (lambda a: a.clone())
    back = (lambda a: a.permute(0, 2, 1, 3).reshape(-1, F, d)) if by_tile else (lambda a: a)
    runs = []
    for _ in range(2):
        w1, m1, v1 = w.clone(), tile(m), tile(v)
        engine.decoder_grad_adam_rows(lists, surv, gd, w1, m1, v1, 1e-2, (0.9, 0.999), 1e-8, 1)
        runs.append((w1, back(m1), back(v1)))
    assert all(torch.equal(a, b) for a, b in zip(*runs))
    w1, m1, v1 = runs[0]
    # the first moments are a tenth of the gradients
    pairs = [(s, t) for s in range(L) for t in range(s, L)]
    want = torch.stack([dense[s].double().t() @ g[t].double() for s, t in pairs])
    size = torch.stack([dense[s].double().abs().t() @ g[t].double().abs() for s, t in pairs])
    got = m1.cpu().double() / (1.0 - torch.tensor(0.9, dtype=torch.float32).double())
    # a lane adds T / 8 products at most, three exchanges add the lanes, two roundings make the moment
    assert bool(((got - want).abs() <= size * (T / 8 + 6) * 2.0 ** -24 + 1e-30).all())
    # the step itself, given the gradient
    w2, m2, v2 = w.clone(), m.clone(), v.clone()
    engine.decoder_weight_grad_adam(lists, surv, gd, w2, m2, v2, 1e-2, (0.9, 0.999), 1e-8, 1)
    assert torch.equal(m1 == 0, m2 == 0)
    assert torch.allclose(v1, v2, rtol=1e-3, atol=1e-6 * float(v2.max()))
    strong = (m2.abs() > 1e-3 * m2.abs().max())            # where the gradient's rounding cannot turn the first step's direction
    assert float((w1 - w2)[:, :, :d][strong].abs().max()) < 1e-4
    assert torch.equal(w1[:, :, d:], w[:, :, d:])


def test_infinities_stay_with_their_features():
    surv, dense, w, m, v, g = _problem(2, 530, 70, 64, 0.05, 3)
    g[1, 520, 7], g[0, 3, 40] = float("inf"), float("nan")
    engine.decoder_grad_adam_rows(engine.feature_lists(surv), surv, g.cuda(), w, m, v, 1e-2, (0.9, 0.999), 1e-8, 1)
    m = m.cpu()                                            # decoders 0->0, 0->1, 1->1
    kept = dense != 0
    assert torch.equal(torch.isnan(m[0, :, 40]), kept[0, 3]) and torch.equal(torch.isinf(m[1, :, 7]), kept[0, 520])
    assert torch.equal(torch.isinf(m[2, :, 7]), kept[1, 520]) and bool(kept[0, 520].any()) and bool(kept[0, 3].any())
    assert torch.equal(m[1, :, 7] > 1e30, dense[0, 520] > 0)
    m[0, :, 40], m[1:, :, 7] = 0.0, 0.0
    assert bool(torch.isfinite(m).all())


def test_which_step_a_float32_shape_takes():
    wanted = lambda T, d, F, L, n: engine.grad_rows_wanted(T, d, F, L, n * T * L, torch.float32)      # noqa: E731
    assert wanted(1024, 768, 6144, 12, 200) == 1 and wanted(1024, 768, 6144, 12, 50) == 1    # 33 and 8.3 entries per list, two tiles
    assert wanted(4096, 768, 6144, 12, 200) == 1 and wanted(4096, 768, 6144, 12, 100) == 0   # 133 and 67, eight tiles
    assert wanted(1500, 1024, 16384, 6, 33) == 2                                             # 3
    assert wanted(1024, 768, 256, 3, 10) == 0 and wanted(1024, 776, 6144, 12, 200) == 0      # too few workgroups; columns
    assert engine.grad_rows_wanted(1024, 768, 6144, 12, 12 * 1024 * 200, torch.bfloat16) == 0


def test_training_takes_the_step_and_keeps_its_state_across_routes():
    # lists of 10.7, 4 and 10.7 entries: LDS tiles, row by row, LDS tiles again, on moments that stay rows; against the kernel row by row
    import crosslayer_coding_amd as cca
    from crosslayer_coding_amd import synth
    runs = []
    for tiles in (True, False):
        model = opt = None
        for step, T in enumerate((683, 256, 683)):
            wl = synth.Workload("rows", step, 4, 512, 1024, T, "float32", k=16)
            if model is None:
                model, x, _ = synth.build_model(wl, torch.device("cuda:0"), 1)
                opt = cca.CLTAdam(model, lr=1e-3)
                opt.tile_decoder_step = tiles
                took = engine.grad_rows_wanted(T, 512, 1024, 4, 4 * T * 16, torch.float32)
                assert took == 1
            gen = torch.Generator().manual_seed(step)
            x = {l: torch.randn(T, 512, generator=gen).cuda() for l in range(4)}
            y = {l: torch.randn(T, 512, generator=gen).cuda() for l in range(4)}
            loss = model.training_step(x, y, opt)
        assert opt._dec_layout == "rows"
        runs.append((float(loss), [t.clone() for t in opt.decoder_moments()], model.decoder_module.packed().clone(), model.state_dict()))
    a, b = runs
    assert abs(a[0] - b[0]) <= 1e-5 * abs(b[0])
    for p, q in zip(a[1], b[1]):
        assert float((p - q).norm() / q.norm()) < 1e-4     # a pre-activation at a cut may change sides once weights differ by a rounding
    assert float((a[2] - b[2]).norm() / b[2].norm()) < 1e-4
    for k, p in a[3].items():                              # parameters are what the packed copy holds
        if k.startswith("decoder_module.decoders.") and k.endswith(".weight"):
            assert float((p - b[3][k]).norm() / b[3][k].norm()) < 1e-4, k


def _called_with(entries, surv, w, m, v, g, out):
    """Both kernels with `entries` in the place of the list's length, on a workspace of that many in the middle of a larger one."""
    from crosslayer_coding_amd import _native as nat
    lib, (ptr, tok, src) = nat.load(), engine.feature_lists(surv)
    L, T, F, d = surv.L, surv.T, surv.F, g.shape[2]
    edges = []
    for need, call in (
            (lib.clt_grad_rows_workspace_bytes(T, d, F, L, entries), lambda ws, n: lib.clt_decoder_grad_adam_rows(
                nat.ptr(ptr), nat.ptr(tok), nat.ptr(src), nat.ptr(surv.val), nat.ptr(g), nat.ptr(w), nat.ptr(m), nat.ptr(v), 0, T, d, F, L,
                entries, 1e-2, 0.9, 0.999, 1e-8, 1, ws, n, nat.current_stream(g.device))),
            (lib.clt_decode_rows_workspace_bytes(T, d, F, L, entries), lambda ws, n: lib.clt_decode_rows(
                nat.ptr(surv.row_ptr), nat.ptr(surv.col), nat.ptr(surv.val), nat.ptr(w), None, None, nat.ptr(out), T, d, F, L, 0, 0, L,
                (1 << L) - 1, entries, ws, n, nat.current_stream(g.device)))):
        room = torch.full((need + (4 << 20),), 0x5A, dtype=torch.uint8, device=g.device)
        assert call(room.data_ptr(), need) == 0
        torch.cuda.synchronize()
        edges.append(bool((room[need:] == 0x5A).all()))
    return edges


def test_lists_longer_than_the_workspace_holds_are_left_alone():
    surv, _, w, m, v, g = _problem(2, 600, 300, 64, 0.05, 5)
    out = torch.full((2, 600, 64), 7.0).cuda()
    w1, m1, v1, out1 = w.clone(), m.clone(), v.clone(), out.clone()
    assert _called_with(surv.capacity - 1, surv, w1, m1, v1, g.cuda(), out1) == [True, True]
    assert torch.equal(w1, w) and torch.equal(m1, m) and torch.equal(v1, v) and torch.equal(out1, out)
    assert _called_with(surv.capacity, surv, w1, m1, v1, g.cuda(), out1) == [True, True]
    assert not torch.equal(w1, w) and not torch.equal(out1, out)


@pytest.mark.parametrize("L,T,F,d,density,by_tile", [(2, 511, 129, 64, 0.05, False), (2, 511, 129, 64, 0.05, True), (3, 700, 140, 96, 0.03, True)])
def test_moments_of_earlier_steps(L, T, F, d, density, by_tile):
    """A later step on moments that are not zero, in both their layouts, against the row kernel: m, v and w differ by what the rounding of
    two gradients makes of them."""
    surv, dense, w, _, _, g = _problem(L, T, F, d, density, T + F)
    lists, gd = engine.feature_lists(surv), g.cuda()
    gen = torch.Generator().manual_seed(7)
    m, v = torch.randn(w.shape[0], F, d, generator=gen).cuda(), (torch.rand(w.shape[0], F, d, generator=gen) + 0.5).cuda()
    tile = (lambda a: a.view(-1, F, d // 8, 8).permute(0, 2, 1, 3).contiguous()) if by_tile else (lambda a: a.clone())
    back = (lambda a: a.permute(0, 2, 1, 3).reshape(-1, F, d)) if by_tile else (lambda a: a)
    lr, step = 1e-2, 5
    w1, m1, v1, w2, m2, v2 = w.clone(), tile(m), tile(v), w.clone(), m.clone(), v.clone()
    engine.decoder_grad_adam_rows(lists, surv, gd, w1, m1, v1, lr, (0.9, 0.999), 1e-8, step)
    engine.decoder_weight_grad_adam(lists, surv, gd, w2, m2, v2, lr, (0.9, 0.999), 1e-8, step)
    m1, v1, w1, m2, v2, w2 = (t.cpu().double() for t in (back(m1), back(v1), w1[:, :, :d], m2, v2, w2[:, :, :d]))
    pairs = [(s, t) for s in range(L) for t in range(s, L)]
    size = torch.stack([dense[s].double().abs().t() @ g[t].double().abs() for s, t in pairs])
    grad = torch.stack([dense[s].double().t() @ g[t].double() for s, t in pairs]).abs()
    ulp = 2.0 ** -23
    off = size * (T / 8 + 6 + T) * ulp / 2                 # of the two sums together
    off_m, off_v = 0.1 * off + m2.abs() * 2 * ulp, 0.001 * (2 * grad * off + off * off) + v2 * 2 * ulp
    assert bool(((m1 - m2).abs() <= off_m).all()) and bool(((v1 - v2).abs() <= off_v).all())
    c1, c2 = 1 - 0.9 ** step, 1 - 0.999 ** step
    root = (v2 / c2).sqrt()
    off_w = lr * (off_m / c1 / root + m2.abs() / c1 / root ** 2 * (off_v / c2 / (2 * root))) + (lr * m2.abs() / c1 / root + w2.abs()) * 4 * ulp
    assert bool(((w1 - w2).abs() <= off_w).all())
    assert float((w2 - w.cpu().double()[:, :, :d]).abs().max()) > 1e-3


def test_training_from_column_tiles_to_lds_tiles_and_back(monkeypatch):
    """Batches of three tiles, of two (twice: the first one stays where the weights are tiled) and three again: 32-byte column tiles, LDS
    tiles on moments that stay in column tiles, and column tiles on a copy of the weights that the step before has put out of date;
    against the kernel row by row."""
    import crosslayer_coding_amd as cca
    from crosslayer_coding_amd import synth
    took, runs = [], []
    for name in ("decoder_weight_grad_adam_tiled", "decoder_grad_adam_rows", "decoder_weight_grad_adam"):
        monkeypatch.setattr(engine, name, lambda *a, _f=getattr(engine, name), _n=name, **kw: took.append(_n) or _f(*a, **kw))
    for tiles in (True, False):
        model = None
        for step, T in enumerate((1100, 683, 683, 1100)):
            wl = synth.Workload("there-and-back", step, 4, 512, 1024, T, "float32", k=16)
            if model is None:
                model, _, _ = synth.build_model(wl, torch.device("cuda:0"), 1)
                opt = cca.CLTAdam(model, lr=1e-3)
                opt.tile_decoder_step = tiles
            gen = torch.Generator().manual_seed(step)
            x = {l: torch.randn(T, 512, generator=gen).cuda() for l in range(4)}
            y = {l: torch.randn(T, 512, generator=gen).cuda() for l in range(4)}
            model.training_step(x, y, opt)
            if tiles:
                assert opt._dec_cols == 8 and took[-1] == ("decoder_grad_adam_rows" if step == 2 else "decoder_weight_grad_adam_tiled")
        runs.append([t.clone() for t in opt.decoder_moments()] + [model.decoder_module.packed().clone()])
    assert took[4:] == ["decoder_weight_grad_adam"] * 4
    for a, b in zip(*runs):
        assert float((a - b).norm() / b.norm()) < 1e-4     # a pre-activation at a cut may change sides once weights differ by a rounding
