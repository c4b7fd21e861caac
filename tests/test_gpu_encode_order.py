"""The order of a float32 product's sum over K: results do not depend on which matrix instruction a kernel is made of."""

import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


def _chain(x, w, b):
    """Fused multiply-adds one after the other, from the bias: 16-byte chunks in pairs, element by element.  A product of two float32
    is exact in float64; the sum rounded to float64 and then to float32 differs from one rounding only where it falls
    within 2^-53 of the middle of two float32, about one step in 2^29."""
    acc = b[:, None, :].expand(-1, x.shape[1], -1).clone()
    for k0 in range(0, x.shape[2], 8):
        for e in range(4):
            for k in (k0 + e, k0 + 4 + e):
                acc = (acc.double() + x[:, :, None, k].double() * w[:, None, :, k].double()).float()
    return acc


@pytest.mark.parametrize("L,T,F,d", [
    (1, 256, 256, 32), (2, 256, 256, 64), (1, 256, 256, 768),      # one tile per layer: K is walked from its first stage
    (2, 300, 512, 96), (3, 257, 264, 160),                         # and so it is in every tile where the stages are odd in number
])
def test_float32_sums_run_over_pairs_of_chunks(L, T, F, d):
    g = torch.Generator().manual_seed(d + T)
    x = torch.randn(L, T, d, generator=g).cuda()
    w = (torch.randn(L, F, d, generator=g) * d ** -0.5).cuda()
    b = torch.randn(L, F, generator=g).cuda()
    got, want = engine.encode(x, w, b), _chain(x, w, b)
    # L T F d steps, one in 2^29 of which may round the other way: less than one expected, three allowed
    assert int((got != want).sum()) <= 3
