"""The gather of all sources' lists as one (clt_decode_thin) against dense products in float64, where its split can go wrong: lists
of 64 and one over (a wavefront's chunk), of 256 and one over (where a workgroup's wavefronts share a token), empty ones, halves of an
odd batch, every shape of a column quarter, and its rule."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat, engine

pytestmark = pytest.mark.gpu


def _lists(L, T, F, per_source, dtype, g):
    """per_source [L, T]: survivors of each (source, token), at random features."""
    keep = torch.zeros(L, T, F, dtype=torch.bool)
    for s in range(L):
        for i in range(T):
            keep[s, i, torch.randperm(F, generator=g)[:int(per_source[s, i])]] = True
    act = torch.where(keep, torch.randn(L, T, F, generator=g), torch.zeros(())).to(dtype)
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(keep.view(L * T, F).sum(1), 0)
    return keep, act, row_ptr


def _decode(keep, act, row_ptr, w, tying, d, bias=None, skip=None, span=None, mask=None, out_f32=False):
    L, T, F = keep.shape
    dev, lib = w.device, nat.load()
    a, b = span or (0, L)
    out = torch.full((L, T, d), 7.0, device=dev, dtype=torch.float32 if out_f32 else act.dtype)
    # one entry more than the lists hold: a list may be empty altogether
    col = torch.cat([keep.view(L * T, F).nonzero()[:, 1].int(), torch.zeros(1, dtype=torch.int32)]).to(dev)
    val = torch.cat([act[keep], torch.zeros(1, dtype=act.dtype)]).to(dev)
    ptr, bias, skip = row_ptr.to(dev), bias if bias is None else bias.to(dev), skip if skip is None else skip.to(dev)
    nat.check(lib.clt_decode_thin(nat.ptr(ptr), nat.ptr(col), nat.ptr(val), nat.ptr(w), nat.ptr(bias), nat.ptr(skip), nat.ptr(out), T, d,
                                  F, L, nat.TYING[tying], a, b, (1 << L) - 1 if mask is None else mask, nat.dtype_code(act.dtype),
                                  1 if out_f32 else 0, nat.current_stream(dev)), "clt_decode_thin")
    return out.cpu()


def _slot(tying, s, t, L):
    return s if tying == "per_source" else s * L - s * (s - 1) // 2 + t - s


@pytest.mark.parametrize("L,T,F,d,dtype,tying,plan,span,mask,out_f32,extra", [
    (1, 1, 40, 512, torch.bfloat16, "none", "few", None, None, False, False),
    (3, 5, 300, 768, torch.bfloat16, "none", "edges", None, None, True, True),       # an odd batch, 64 / 65 / 256 / 257 per token
    (3, 9, 300, 1024, torch.bfloat16, "per_source", "edges", None, None, True, False),
    (2, 33, 700, 2048, torch.bfloat16, "none", "edges", None, None, False, True),
    (4, 7, 300, 512, torch.float16, "none", "edges", None, None, True, True),
    (3, 8, 300, 512, torch.float32, "none", "edges", None, None, False, True),
    (3, 11, 300, 768, torch.float32, "per_source", "edges", None, None, False, False),
    (2, 6, 900, 1024, torch.float32, "none", "edges", None, None, False, True),
    (6, 10, 200, 768, torch.bfloat16, "none", "edges", (2, 5), 0b101011, True, True),  # some targets, some sources
    (3, 10, 200, 512, torch.bfloat16, "none", "edges", None, 0, True, True),           # no source at all
    (64, 3, 64, 512, torch.bfloat16, "per_source", "few", (60, 64), None, True, False),  # as many sources as lanes
])
def test_decode_thin_against_dense_products(L, T, F, d, dtype, tying, plan, span, mask, out_f32, extra):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(L * T + d)
    n = torch.randint(0, 4, (L, T), generator=g)
    if plan == "edges":                        # totals of the first tokens, dealt over the sources in unequal shares
        for i, total in enumerate([64, 65, 256, 257, 128, 0][:T]):
            n[:, i] = 0
            n[0, i] = min(F, total // 3 if L > 1 else total)
            n[1 % L, i] += total - int(n[0, i])
        n = n.clamp(max=F)
        n[:, T - 1] = min(F, 200)              # more than 256 in all from the second target on
    keep, act, row_ptr = _lists(L, T, F, n, dtype, g)
    n_dec = L if tying == "per_source" else L * (L + 1) // 2
    w = engine.alloc_packed(n_dec, F, d, dtype, dev)
    w[:, :, :d] = torch.randn(n_dec, F, d, generator=g).to(dev, dtype)
    bias = torch.randn(L, d, generator=g) if extra else None
    skip = torch.randn(L, T, d, generator=g) if extra else None
    got, again = (_decode(keep, act, row_ptr, w, tying, d, bias, skip, span, mask, out_f32) for _ in range(2))
    assert torch.equal(got, again)
    a, b = span or (0, L)
    mask = (1 << L) - 1 if mask is None else mask
    wc, x = w.cpu()[:, :, :d].double(), act.double()
    for t in range(L):
        if not a <= t < b:
            assert bool((got[t] == 7.0).all())              # not asked for
            continue
        ref = torch.zeros(T, d, dtype=torch.float64)
        if extra:
            ref = bias[t].double() + skip[t].double()
        mag, n_t = ref.abs() if not extra else bias[t].double().abs() + skip[t].double().abs(), 0
        for s in range(t + 1):
            if (mask >> s) & 1:
                m = wc[_slot(tying, s, t, L)]
                ref, mag, n_t = ref + x[s] @ m, mag + x[s].abs() @ m.abs(), n_t + keep[s].sum(1, keepdim=True)
        # products of 16 bits are exact in fp32; one rounding per multiply-add or addition, each at most 2^-24 of what has been
        # summed, and one of the result where it is stored as bf16: half of a last place of 8 significant bits, 2^-8 of it at most
        tol = (n_t + 8.0) * 2.0 ** -24 * mag
        if not out_f32 and dtype == torch.bfloat16:
            tol = tol + (ref.abs() + tol) * 2.0 ** -8
        assert bool(((got[t].double() - ref).abs() <= tol).all())


def test_decode_thin_keeps_values_that_are_not_finite_to_their_tokens():
    dev = torch.device("cuda:0")
    L, T, F, d = 2, 6, 64, 512
    g = torch.Generator().manual_seed(2)
    keep, act, row_ptr = _lists(L, T, F, torch.full((L, T), 3), torch.bfloat16, g)
    w = engine.alloc_packed(3, F, d, torch.bfloat16, dev)
    w[:, :, :d] = torch.randn(3, F, d, generator=g).to(dev, torch.bfloat16)
    bad = int(keep[0, 2].nonzero()[0])
    w[0, bad, 5], w[0, bad, 300] = float("inf"), float("nan")
    act[1, 4] = torch.where(keep[1, 4], torch.full((), float("inf"), dtype=torch.bfloat16), act[1, 4])
    got = _decode(keep, act, row_ptr, w, "none", d, out_f32=True)
    hit = keep[0, :, bad]
    assert bool(torch.isinf(got[0, hit, 5]).all()) and bool(torch.isnan(got[0, hit, 300]).all())
    assert bool(torch.isfinite(got[0, ~hit]).all())
    fine = [i for i in range(d) if i not in (5, 300)]
    assert bool(torch.isfinite(got[0][hit][:, fine]).all())
    assert bool(torch.isfinite(got[1][[0, 1, 2, 3, 5]]).all()) and not bool(torch.isfinite(got[1, 4]).any())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_decode_thin_is_chosen_and_agrees_with_the_gather(monkeypatch, dtype):
    dev, lib = torch.device("cuda:0"), nat.load()
    L, T, F, d, k = 8, 1200, 8192, 768, 24
    wanted = lambda *a: lib.clt_decode_thin_wanted(*a, nat.dtype_code(dtype))
    assert wanted(T, d, F, L, L, T * k, nat.TYING["none"]) == 1
    assert wanted(T, d, F, L, L, T * k, nat.TYING["per_target"]) == 0
    assert wanted(T, d + 32, F, L, L, T * k, nat.TYING["none"]) == 0
    assert wanted(T, d, 2 ** 27, L, L, T * k, nat.TYING["none"]) == 0       # row numbers beyond 31 bits
    assert wanted(T, d, F, L, L, L * T * 200, nat.TYING["none"]) == 0       # lists that are not thin
    g = torch.Generator().manual_seed(3)
    surv = engine.batchtopk_select(torch.randn(L, T, F, generator=g).to(dev, dtype), k, True)
    assert surv.status is None and surv.capacity == T * k
    w = engine.alloc_packed(L * (L + 1) // 2, F, d, dtype, dev)
    w[:, :, :d] = torch.randn(L * (L + 1) // 2, F, d, generator=g).to(dev, dtype)
    ws, ran = engine.Workspace(dev), []
    thin = lib.clt_decode_thin
    monkeypatch.setattr(lib, "clt_decode_thin", lambda *a: ran.append(1) or thin(*a))
    got = engine.decode_sparse(surv, w, "none", d, ws=ws, out_f32=True)
    assert ran == [1]
    engine.decode_sparse(engine.SurvivorList(surv.row_ptr, surv.col, surv.val, T, F, L, dtype), w, "none", d, ws=ws)
    assert ran == [1]                            # a list of unknown origin, whose length says nothing about a row
    monkeypatch.setattr(lib, "clt_decode_thin_wanted", lambda *a: 0)
    ref = engine.decode_sparse(surv, w, "none", d, ws=ws, out_f32=True)
    assert ran == [1] and float((got - ref).norm() / ref.norm()) < 1e-6     # fp32 sums in another order


@pytest.mark.parametrize("L,T,F,d,dtype,tying,out_f32,extra", [
    (3, 40, 9000, 512, torch.bfloat16, "none", True, True),
    (2, 17, 9000, 768, torch.bfloat16, "per_source", False, False),
    (3, 33, 8300, 512, torch.float16, "none", True, False),
    (2, 19, 8300, 768, torch.float32, "none", False, True),
])
def test_decode_thin_of_the_longest_lists(L, T, F, d, dtype, tying, out_f32, extra):
    """Lists around 8192 entries, above which a kernel of its own sums them: one entry more and one less, those that cross the line
    with a later source, two in one sixteenth of the batch, and the last token."""
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(T)
    n = torch.randint(0, 4, (L, T), generator=g)
    n[:, 1] = torch.tensor([8192] + [0] * (L - 1))
    n[:, 2] = torch.tensor([8193] + [0] * (L - 1))
    n[:, 3] = torch.tensor([8191] + [1] * (L - 1))         # 8192 at target 1, at target 2 one more
    n[:, T // 2] = F
    n[:, T - 1] = torch.tensor([0, 8200] + [5] * (L - 2))
    keep, act, row_ptr = _lists(L, T, F, n, dtype, g)
    n_dec = L if tying == "per_source" else L * (L + 1) // 2
    w = engine.alloc_packed(n_dec, F, d, dtype, dev)
    w[:, :, :d] = torch.randn(n_dec, F, d, generator=g).to(dev, dtype)
    bias = torch.randn(L, d, generator=g) if extra else None
    skip = torch.randn(L, T, d, generator=g) if extra else None
    got, again = (_decode(keep, act, row_ptr, w, tying, d, bias, skip, out_f32=out_f32) for _ in range(2))
    assert torch.equal(got, again)
    wc, x = w[:, :, :d].double(), act.double().to(dev)
    for t in range(L):
        zero = torch.zeros(T, d, dtype=torch.float64, device=dev)
        ref, mag, n_t = zero, zero, 0
        if extra:                                           # two summands: they may cancel
            ref = bias[t].double().to(dev) + skip[t].double().to(dev)
            mag = bias[t].double().abs().to(dev) + skip[t].double().abs().to(dev)
        for s in range(t + 1):
            m = wc[_slot(tying, s, t, L)]
            ref, mag, n_t = ref + x[s] @ m, mag + x[s].abs() @ m.abs(), n_t + keep[s].sum(1, keepdim=True).to(dev)
        tol = (n_t + 8.0) * 2.0 ** -24 * mag                # as above
        if not out_f32 and dtype == torch.bfloat16:
            tol = tol + (ref.abs() + tol) * 2.0 ** -8
        assert bool(((got[t].double().to(dev) - ref).abs() <= tol).all()), t


def test_decode_thin_of_a_long_list_keeps_values_that_are_not_finite():
    dev = torch.device("cuda:0")
    L, T, F, d = 1, 18, 8300, 512
    g = torch.Generator().manual_seed(2)
    n = torch.full((L, T), 3)
    n[0, 4], n[0, 5] = 8195, 8197                          # no whole number of eights, nor of 64s
    keep, act, row_ptr = _lists(L, T, F, n, torch.bfloat16, g)
    w = engine.alloc_packed(1, F, d, torch.bfloat16, dev)
    w[:, :, :d] = torch.randn(1, F, d, generator=g).to(dev, torch.bfloat16)
    bad = int((keep[0, 4] & ~keep[0, 5]).nonzero()[0])
    w[0, bad, 5], w[0, 0, 7] = float("inf"), float("nan")   # row 0 is what the places past the end refer to
    keep[0, :, 0] = False
    act[0, :, 0] = 0
    row_ptr[1:] = torch.cumsum(keep.view(T, F).sum(1), 0)
    got = _decode(keep, act, row_ptr, w, "none", d, out_f32=True)
    hit = keep[0, :, bad]
    assert bool(hit[4]) and not bool(hit[5])
    assert bool(torch.isinf(got[0, hit, 5]).all()) and bool(torch.isfinite(got[0, ~hit]).all())
    assert bool(torch.isfinite(got[0][:, [i for i in range(d) if i != 5]]).all())


@pytest.mark.parametrize("hint", [20000, 400000])
def test_a_threshold_list_that_outgrew_its_hint_is_decoded(monkeypatch, hint):
    """The hint chooses the gather for thin lists; whether the list is one is decided on the device."""
    dev, lib = torch.device("cuda:0"), nat.load()
    L, T, F, d = 6, 1500, 4096, 768
    g = torch.Generator().manual_seed(4)
    pre = torch.randn(L, T, F, generator=g).to(dev, torch.bfloat16)
    exact = engine.batchtopk_select(pre, 250, True)         # 375 000 entries
    surv = engine.SurvivorList(exact.row_ptr, exact.col, exact.val, T, F, L, torch.bfloat16,
                               torch.zeros(1, dtype=torch.int32, device=dev), hint, True)
    w = engine.alloc_packed(L * (L + 1) // 2, F, d, torch.bfloat16, dev)
    w[:, :, :d] = torch.randn(L * (L + 1) // 2, F, d, generator=g).to(dev, torch.bfloat16)
    monkeypatch.setattr(lib, "clt_decode_thin_wanted", lambda *a: 1)
    got = engine.decode_sparse(surv, w, "none", d, ws=engine.Workspace(dev), out_f32=True)
    monkeypatch.setattr(lib, "clt_decode_thin_wanted", lambda *a: 0)
    ref = engine.decode_sparse(exact, w, "none", d, ws=engine.Workspace(dev), out_f32=True)
    assert float((got - ref).norm() / ref.norm()) < 1e-6    # fp32 sums in another order
