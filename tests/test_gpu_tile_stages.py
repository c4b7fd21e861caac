"""The batches of a stage (spmm.h): groups with none, one and many batches in every order, stages that begin and end at each place
of a quad of records, at four groups per wavefront."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat, engine

pytestmark = pytest.mark.gpu


def _lists(L, T, F, densities, dev, seed):
    """Activations whose density in each (layer, 16 tokens, 512 features) is one of `densities`."""
    g = torch.Generator(dev).manual_seed(seed)
    pick = torch.randint(len(densities), (L, T // 16, F // 512), generator=g, device=dev)
    p = torch.tensor(densities, device=dev)[pick].repeat_interleave(16, 1).repeat_interleave(512, 2)
    act = torch.where(torch.rand(L, T, F, generator=g, device=dev) < p, torch.randn(L, T, F, generator=g, device=dev), 0.0).bfloat16()
    nz = act.view(L * T, F) != 0
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32, device=dev)
    row_ptr[1:] = torch.cumsum(nz.sum(1), 0)
    return act, row_ptr, nz.nonzero()[:, 1].int(), act.view(L * T, F)[nz], g


@pytest.mark.parametrize("densities", [
    [0.0, 0.0006, 0.004, 0.02], [0.0, 0.0, 0.0, 0.0, 0.0002], [0.009], [0.0, 0.05],
])
def test_stages_of_four_groups(densities):
    dev = torch.device("cuda:0")
    L, T, F, d = 4, 4096, 2048, 2048           # 512 workgroups of sixteen wavefronts with four groups each
    act, row_ptr, col, val, g = _lists(L, T, F, densities, dev, len(densities))
    w = torch.randn(L, F, d, generator=g, device=dev).bfloat16()
    slab = engine.alloc_packed(L, F, d, torch.bfloat16, dev)
    slab[:, :, :d] = w
    lib = nat.load()
    ws = torch.full((lib.clt_decode_tiles_workspace_bytes(T, d, F, L, L, col.numel()),), 0xFF, dtype=torch.uint8, device=dev)
    out = torch.empty(L, T, d, device=dev)
    c, v = torch.cat([col, col.new_zeros(1)]), torch.cat([val, val.new_zeros(1)])
    nat.check(lib.clt_decode_tiles(nat.ptr(row_ptr), nat.ptr(c), nat.ptr(v), nat.ptr(slab), None, None, nat.ptr(out), T, d, F, L,
                                   nat.TYING["per_source"], 0, L, (1 << L) - 1, nat.dtype_code(torch.bfloat16), 1, col.numel(), nat.ptr(ws),
                                   ws.numel(), nat.current_stream(dev)), "clt_decode_tiles")
    ref, mag = torch.zeros(T, d, dtype=torch.float64, device=dev), torch.zeros(T, d, dtype=torch.float64, device=dev)
    n = torch.zeros(T, 1, device=dev)
    for t in range(L):
        ref += act[t].double() @ w[t].double()
        mag += act[t].double().abs() @ w[t].double().abs()
        n += (act[t] != 0).sum(1, keepdim=True)
        # exact products; each addition is off by at most 2^-23 of what has been summed
        assert ((out[t].double() - ref).abs() <= (n + 2) * 2.0 ** -23 * mag).all(), t


@pytest.mark.parametrize("densities", [[0.0, 0.0006, 0.004, 0.02], [0.0, 0.0, 0.0, 0.0002], [0.009]])
def test_gradient_stages_begin_inside_a_quad(densities):
    dev = torch.device("cuda:0")
    L, T, F, d = 3, 2560, 1536, 128
    act, row_ptr, col, val, g = _lists(L, T, F, densities, dev, 7 + len(densities))
    surv = engine.SurvivorList(row_ptr, col, val, T, F, L, torch.bfloat16)
    gm = torch.randn(L, T, d, generator=g, device=dev).bfloat16()
    ws = engine.Workspace(dev)
    ws.get("grad_tiles", nat.load().clt_grad_tiles_workspace_bytes(T, d, F, L, surv.capacity)).fill_(0xFF)
    got = engine.decoder_weight_grad(engine.feature_lists(surv, ws), surv, gm, "none", ws=ws)
    slot = 0
    for s in range(L):
        for t in range(s, L):
            a = act[s].double().t()
            bound = ((act[s] != 0).sum(0).double().unsqueeze(1) + 1) * 2.0 ** -23 * (a.abs() @ gm[t].double().abs())
            assert ((got[slot].double() - a @ gm[t].double()).abs() <= bound).all(), (s, t)
            slot += 1
