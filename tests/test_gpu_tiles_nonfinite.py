"""Infinities and NaNs in the operands of the products from LDS tiles (decodes and weight gradient) reach the
output rows whose lists refer to them and no others, although a batch's 16 rows are multiplied together."""
import pytest
import torch

from crosslayer_coding_amd import engine
from crosslayer_coding_amd import _native as nat

pytestmark = pytest.mark.gpu
L, T, F, d, K = 3, 200, 1100, 128, 12


def _lists(dtype):
    g = torch.Generator().manual_seed(5)
    keep = torch.zeros(L, T, F, dtype=torch.bool)
    keep.scatter_(2, torch.rand(L, T, F, generator=g).topk(K, dim=2).indices, True)
    act = torch.where(keep, torch.rand(L, T, F, generator=g) + 0.5, torch.zeros(())).to(dtype)
    ptr = torch.arange(0, L * T * K + 1, K, dtype=torch.int32).cuda()
    surv = engine.SurvivorList(ptr, keep.view(L * T, F).nonzero()[:, 1].int().cuda(), act[keep].cuda(), T, F, L, dtype)
    return g, keep, act, surv


def _check(got, ref, mag):
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    fin = ref.isfinite()
    # bf16 rounding of the result; sums of less than 256 exact products in fp32
    assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -15 * mag)[fin].all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode(dtype, monkeypatch):
    g, keep, act, surv = _lists(dtype)
    monkeypatch.setattr(nat.load(), "clt_decode_tiles_wanted", lambda *a: 1)
    n_dec = L * (L + 1) // 2
    w = engine.alloc_packed(n_dec, F, d, dtype, torch.device("cuda:0"))
    wc = torch.randn(n_dec, F, d, generator=g).to(dtype)
    wc[0, 0, :70] = float("inf")                  # the row that the fills of a batch refer to, in both column parts
    wc[1, 512, 3], wc[2, 1099, 100], wc[4, 700, 64] = float("nan"), -float("inf"), float("inf")
    w[:, :, :d] = wc.cuda()
    bias = torch.randn(L, d, generator=g)
    got = engine.decode_sparse(surv, w, "none", d, bias_sum=bias.cuda(), ws=engine.Workspace(torch.device("cuda:0"))).cpu().double()
    for t in range(L):
        ref, mag = bias[t].double().expand(T, d).clone(), bias[t].double().abs().expand(T, d).clone()
        for s in range(t + 1):
            m = wc[s * L - s * (s - 1) // 2 + t - s].double()
            for tok in range(T):
                f = keep[s, tok]
                ref[tok] += act[s, tok, f].double() @ m[f]
                mag[tok] += act[s, tok, f].double().abs() @ m[f].abs()
        _check(got[t], ref, mag)


@pytest.mark.parametrize("adam", [False, True])
def test_weight_gradient(adam):
    g, keep, act, surv = _lists(torch.bfloat16)
    gm = torch.randn(L, T, d, generator=g).bfloat16()
    gm[0, 0, 5], gm[1, 17, 70], gm[2, 199, 0] = float("inf"), float("nan"), -float("inf")
    ws = engine.Workspace(torch.device("cuda:0"))
    lists = engine.feature_lists(surv, ws)
    assert engine.grad_tiles_supported(T, d, F, L, surv.capacity, torch.bfloat16)
    n_dec = L * (L + 1) // 2
    if adam:
        w = engine.alloc_packed(n_dec, F, d, torch.bfloat16, torch.device("cuda:0"))
        w[:, :, :d] = 1.0
        m, v = torch.zeros(n_dec, F, d, device="cuda"), torch.zeros(n_dec, F, d, device="cuda")
        engine.decoder_grad_adam_tiles(lists, surv, gm.cuda(), w, m, v, 1e-2, (0.0, 0.0), 1e-8, 1, ws=ws)      # m is the gradient
        got = m.cpu().double()
        step = got.sign() * got.abs().clamp(max=1)
        live = got.isfinite()
        assert bool((w[:, :, :d].cpu().double()[live & (got.abs() > 1e-3)] - (1.0 - 1e-2 * step.sign())[live & (got.abs() > 1e-3)]).abs().max() < 4e-3)
        assert bool((w[:, :, :d].cpu()[live & (got == 0)] == 1.0).all())
    else:
        got = engine.decoder_weight_grad(lists, surv, gm.cuda(), "none", ws=ws).cpu().double()
    slot = 0
    for s in range(L):
        for t in range(s, L):
            ref, mag = torch.zeros(F, d, dtype=torch.float64), torch.zeros(F, d, dtype=torch.float64)
            for f in range(F):
                r = keep[s, :, f]
                ref[f] = act[s, r, f].double() @ gm[t, r].double()
                mag[f] = act[s, r, f].double().abs() @ gm[t, r].double().abs()
            _check(got[slot], ref, mag)
            slot += 1


def test_decode_rows(monkeypatch):
    """The float32 decode multiplies the places that fill a record up (a run's last entry once more, value 0) with that entry's
    decoder row: an infinity there stays an infinity."""
    g, keep, act, surv = _lists(torch.float32)
    monkeypatch.setattr(nat.load(), "clt_decode_rows_wanted", lambda *a: 1)
    n_dec = L * (L + 1) // 2
    w = engine.alloc_packed(n_dec, F, d, torch.float32, torch.device("cuda:0"))
    wc = torch.randn(n_dec, F, d, generator=g)
    for i, tok in enumerate((0, 17, 199)):        # the last features of a token's runs, which are shorter than a record
        kept = keep[0, tok].nonzero()[:, 0]
        for c in range(3):
            wc[i, kept[kept < 512 * (c + 1)][-1], 5 + 40 * c] = float("inf") * (-1) ** c
    wc[1, 512, 3], wc[4, 700, 64] = float("nan"), float("inf")
    w[:, :, :d] = wc.cuda()
    bias = torch.randn(L, d, generator=g)
    got = engine.decode_sparse(surv, w, "none", d, bias_sum=bias.cuda(), ws=engine.Workspace(torch.device("cuda:0"))).cpu().double()
    for t in range(L):
        ref, mag = bias[t].double().expand(T, d).clone(), bias[t].double().abs().expand(T, d).clone()
        for s in range(t + 1):
            m = wc[s * L - s * (s - 1) // 2 + t - s].double()
            for tok in range(T):
                f = keep[s, tok]
                ref[tok] += act[s, tok, f].double() @ m[f]
                mag[tok] += act[s, tok, f].double().abs() @ m[f].abs()
        assert torch.equal(got[t].isnan(), ref.isnan()) and torch.equal(got[t].isinf(), ref.isinf()) and bool(ref.isinf().any())
        fin = ref.isfinite()
        # at most K sources' entries and eight sums more, each addition off by at most 2^-24 of what has been summed
        assert bool(((got[t] - ref).abs() <= (L * K + 16) * 2.0 ** -24 * mag)[fin].all())
