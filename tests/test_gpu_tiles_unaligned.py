"""Operands that begin at any element, which the gathers take, are not refused where the shapes would go to the kernels over LDS
tiles (those want 16-byte addresses)."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat
from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu
L, T, F, d, K = 2, 64, 1024, 128, 10


def _surv(dtype):
    g = torch.Generator().manual_seed(2)
    keep = torch.zeros(L, T, F, dtype=torch.bool)
    keep.scatter_(2, torch.rand(L, T, F, generator=g).topk(K, dim=2).indices, True)
    act = torch.where(keep, torch.rand(L, T, F, generator=g) + 0.5, torch.zeros(())).to(dtype)
    ptr = torch.arange(0, L * T * K + 1, K, dtype=torch.int32).cuda()
    return g, engine.SurvivorList(ptr, keep.view(L * T, F).nonzero()[:, 1].int().cuda(), act[keep].cuda(), T, F, L, dtype)


def _shifted(x):
    """The same tensor from the second 32-bit word of its storage on."""
    skip = 4 // x.element_size()
    out = torch.empty(x.numel() + skip, dtype=x.dtype, device="cuda")[skip:].view(x.shape)
    assert out.data_ptr() % 16 == 4 and out.is_contiguous()
    return out.copy_(x)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_decode(dtype, monkeypatch):
    g, surv = _surv(dtype)
    for name in ("clt_decode_tiles_wanted", "clt_decode_rows_wanted"):
        monkeypatch.setattr(nat.load(), name, lambda *a: 1)
    w = engine.alloc_packed(3, F, d, dtype, torch.device("cuda:0"))
    w[:, :, :d] = torch.randn(3, F, d, generator=g).to(dtype).cuda()
    bias, skip = torch.randn(L, d, generator=g), torch.randn(L, T, d, generator=g)
    ws = engine.Workspace(torch.device("cuda:0"))
    ref = engine.decode_sparse(surv, w, "none", d, bias_sum=bias.cuda(), skip_add=skip.cuda(), ws=ws, out_f32=True)
    for b, s in ((_shifted(bias), skip.cuda()), (bias.cuda(), _shifted(skip))):
        got = engine.decode_sparse(surv, w, "none", d, bias_sum=b, skip_add=s, ws=ws, out_f32=True)
        # at most 22 terms below 10 in another order
        assert float((got - ref).abs().max()) <= 22 * 2.0 ** -23 * 200


def test_weight_gradient():
    g, surv = _surv(torch.bfloat16)
    gm = torch.randn(L, T, d, generator=g).bfloat16()
    ws = engine.Workspace(torch.device("cuda:0"))
    lists = engine.feature_lists(surv, ws)
    assert engine.grad_tiles_supported(T, d, F, L, surv.capacity, torch.bfloat16)
    ref = engine.decoder_weight_grad(lists, surv, gm.cuda(), "none", ws=ws)
    got = engine.decoder_weight_grad(lists, surv, _shifted(gm), "none", ws=ws)
    assert float((got - ref).abs().max()) <= T * 2.0 ** -23 * 200
