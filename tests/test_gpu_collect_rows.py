"""The ordered write of the candidates that the encoder's epilogue collects (k_tile_count, k_tile_emit) against the selection on
stored pre-activations: 64 entries at a time, 128 in flight per extent, 2 or 8 segments per wavefront.  Rows that hold whole segments
(a run longer than a wavefront, rows cut by the 64s), rows with none, batches and features that are no whole number of
tiles, and ties that a row's allotment cuts, all in small whole numbers, so that both sides have the same pre-activations."""
import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


def _operands(L, T, d, F, dtype, heavy, g):
    dev = torch.device("cuda:0")
    x = torch.randint(-1, 2, (L, T, d), generator=g).float()
    w = torch.randint(-1, 2, (L, F, d), generator=g).float()
    if heavy:                                   # tokens that reach the threshold at almost every feature, and some at none
        w[:, :, 0] = 1.0
        x[:, ::37, 0] = 100.0
        x[:, 5::41, 0] = -100.0
    b = torch.randint(-2, 3, (L, F), generator=g).float()
    return x.to(dev, dtype), w.to(dev, dtype), b.to(dev, dtype)


def _same(got, ref):
    n = int(ref.row_ptr[-1])
    assert torch.equal(got.row_ptr.cpu(), ref.row_ptr.cpu())
    assert torch.equal(got.col[:n].cpu(), ref.col[:n].cpu()) and torch.equal(got.val[:n].cpu(), ref.val[:n].cpu())


SHAPES = [
    (1, 256, 64, 256, 5, False),
    (2, 257, 64, 1032, 9, True),                # a shifted token tile of one row, 9 segments in 16 bits, the last one ragged
    (2, 300, 64, 2304, 40, True),
    (1, 511, 128, 520, 130, True),              # a quarter of the features kept
    (3, 640, 64, 4096, 3, True),
    (8, 1030, 64, 53000, 4, True),              # extents enough for eight of them to a wavefront (two in the others)
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("L,T,d,F,k,heavy", SHAPES)
def test_collected_topk_is_the_selection_of_stored_ones(L, T, d, F, k, heavy, dtype):
    x, w, b = _operands(L, T, d, F, dtype, heavy, torch.Generator().manual_seed(T + F))
    assert engine.encode_collect_supported(x, w, b, k)
    pre = engine.encode(x, w, b)
    ws = engine.Workspace(x.device)
    got = engine.collect_select(engine.encode_collect(x, w, b, k, torch.empty_like(pre), ws))
    _same(got, engine.batchtopk_select(pre, k, False))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("L,T,d,F,k,heavy", SHAPES)
def test_collected_threshold_list_is_that_of_stored_ones(L, T, d, F, k, heavy, dtype):
    g = torch.Generator().manual_seed(T + F)
    x, w, b = _operands(L, T, d, F, dtype, heavy, g)
    theta = (torch.randint(12, 22, (L, F), generator=g).float() * (d / 64) ** 0.5).floor().to(x.device, dtype)
    pre = engine.encode(x, w, b)
    got = engine.encode_threshold(x, w, b, theta, engine.Workspace(x.device), density_ppm=200000)
    assert got is not None
    keep = pre >= theta[:, None]
    n = int(got.row_ptr[-1])
    assert n == int(keep.sum()) and torch.equal(torch.diff(got.row_ptr.long()), keep.sum(2).flatten())
    assert torch.equal(got.col[:n].long(), keep.view(L * T, F).nonzero()[:, 1]) and torch.equal(got.val[:n], pre[keep])
