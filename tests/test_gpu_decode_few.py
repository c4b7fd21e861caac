"""The gather decode of launches with few rows (16 survivors in flight, one wavefront per workgroup) gives the bits of a long
launch: the same rows, alone and as the first rows of a batch with more rows than the rule allows."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,d,F,dtype,tying", [
    (3, 768, 300, torch.float32, "none"), (4, 768, 260, torch.bfloat16, "none"), (3, 520, 200, torch.float16, "per_source"),
    (2, 1020, 130, torch.float32, "per_target"), (5, 48, 100, torch.bfloat16, "per_target"), (64, 64, 100, torch.float32, "per_source"),
    (3, 1024, 150, torch.float32, "none"), (2, 1280, 150, torch.bfloat16, "none"),
    (2, 1536, 130, torch.bfloat16, "none"), (2, 1792, 130, torch.bfloat16, "none"), (2, 1792, 130, torch.float16, "none"),
    (2, 2000, 130, torch.bfloat16, "none"),                  # three pieces of 16 bytes a lane: alone, and with a half and a whole one more
])
@pytest.mark.parametrize("T,span,mask", [(1, None, None), (16, None, None), (5, (1, 2), 0b11), (3, None, 0)])
def test_few_rows_and_many(L, d, F, dtype, tying, T, span, mask):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(T + d)
    n_dec = L * (L + 1) // 2 if tying == "none" else L
    w = engine.alloc_packed(n_dec, F, d, dtype, dev)
    w[:, :, :d] = torch.randn(n_dec, F, d, generator=g).to(dtype).to(dev)
    keep = torch.rand(L, T, F, generator=g) < 0.2
    keep[:, 0, :] = True                                     # several chunks of 64
    keep[1] = False                                          # a source without survivors
    vals = torch.randn(L, T, F, generator=g).to(dtype)
    bias, outs = torch.randn(L, d, generator=g).to(dev), []
    a, b = span or (0, L)
    for rows in (T, 1024 // (b - a) + 8):
        full = torch.zeros(L, rows, F, dtype=torch.bool)
        full[:, :T] = keep
        ptr = torch.zeros(L * rows + 1, dtype=torch.int32)
        ptr[1:] = torch.cumsum(full.view(L * rows, F).sum(1), 0)
        surv = engine.SurvivorList(ptr.to(dev), full.view(L * rows, F).nonzero()[:, 1].int().to(dev), vals[keep].to(dev), rows, F, L, dtype)
        outs.append(engine.decode_sparse(surv, w, tying, d, bias_sum=bias, t_begin=a, t_end=b, src_mask=mask, ws=None,
                                         out_f32=True)[a:b, :T].clone())
    assert torch.equal(outs[0], outs[1])


def test_a_narrower_row_is_no_slower():
    """bf16, d = 1792 against 1920: 16 survivors in flight took more registers than there are for the narrower row alone (2.3
    times the wider one's time).  The best of ten launches each, allowed 1.4 times."""
    dev, L, T, F, k = torch.device("cuda:0"), 4, 32, 1024, 100
    g = torch.Generator(device=dev).manual_seed(1)
    col = (torch.rand(L * T, k, generator=g, device=dev) * (F // k)).int() + torch.arange(k, device=dev, dtype=torch.int32) * (F // k)
    surv = engine.SurvivorList(torch.arange(0, L * T * k + 1, k, dtype=torch.int32, device=dev), col.reshape(-1),
                               torch.randn(L * T * k, generator=g, device=dev).bfloat16(), T, F, L, torch.bfloat16)
    ms = {}
    for d in (1792, 1920):
        w = engine.alloc_packed(L * (L + 1) // 2, F, d, torch.bfloat16, dev)
        w[:, :, :d] = torch.randn(F, d, generator=g, device=dev).bfloat16()
        out, best = torch.empty(L, T, d, dtype=torch.bfloat16, device=dev), []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                engine.decode_sparse(surv, w, "none", d, out=out)
            b.record()
            torch.cuda.synchronize()
            best.append(a.elapsed_time(b))
        ms[d] = min(best[2:])
    assert ms[1792] <= 1.4 * ms[1920], ms
