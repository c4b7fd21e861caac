"""Gradients of many parameters rounded to bf16 in one launch (clt_cast_many) are torch's casts bit for bit: whole and ragged pieces, sources
that begin at any float, more tensors than a launch holds, empty ones among them."""
import ctypes

import pytest
import torch

from crosslayer_coding_amd import _native as nat
from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    [(3, 1)], [(1, 8192)], [(2, 8191), (5, 3)], [(2, 8193), (3, 16384)], [(4, 100, 130), (4, 100), (10, 130), (10, 30, 30)], [(130, 77), (1, 5)],
])
def test_families(shapes):
    g = torch.Generator().manual_seed(len(shapes))
    families = [torch.randn(shape, generator=g).cuda() for shape in shapes]
    for f in families:
        f.view(-1)[0], f.view(-1)[-1] = float("inf"), 3.39e38                # (the largest finite numbers round to infinity)
        f.view(-1)[f.numel() // 2] = float("nan")
    for f, parts in zip(families, engine.parameter_gradients(families, torch.bfloat16)):
        assert len(parts) == f.shape[0]
        for got, want in zip(parts, f.bfloat16().unbind(0)):
            assert got.shape == want.shape and got.untyped_storage().nbytes() == 2 * got.numel()
            nan = want.isnan()
            assert torch.equal(got.isnan(), nan) and torch.equal(got.masked_fill(nan, 0), want.masked_fill(nan, 0))


def test_empty_tensors_and_edges():
    sizes = [0, 5, 0, 8192, 0, 0, 20000, 0]
    source = torch.randn(sum(sizes) + 3).cuda()[3:]                          # begins at no 16-byte address
    room = torch.full((sum(sizes) + 64 * len(sizes),), 7.0, dtype=torch.bfloat16).cuda()
    n = len(sizes)
    starts, ends = [sum(sizes[:i]) for i in range(n)], [sum(sizes[:i]) + 32 * i for i in range(n)]
    a = (ctypes.c_void_p * n)(*[source.data_ptr() + 4 * s for s in starts])
    b = (ctypes.c_void_p * n)(*[room.data_ptr() + 2 * e for e in ends])
    c = (ctypes.c_int64 * n)(*sizes)
    code = nat.load().clt_cast_many(ctypes.addressof(a), ctypes.addressof(b), ctypes.addressof(c), n, nat.CLT_BF16, nat.current_stream(room.device))
    assert code == 0
    want = torch.full_like(room, 7.0)
    for s, e, size in zip(starts, ends, sizes):
        want[e:e + size] = source[s:s + size].bfloat16()
    assert torch.equal(room, want)
