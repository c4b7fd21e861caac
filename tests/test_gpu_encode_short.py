"""Encoder projection of batches shorter than one matrix tile (k_encode_short), against float64."""

import pytest
import torch

from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu

# unit roundoff of the one rounding at the end
ROUND = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dtype", list(ROUND), ids=lambda t: str(t).split(".")[1])
@pytest.mark.parametrize("T,d,F,L,bias", [
    (1, 64, 8, 1, True),           # one stage of K, one quad of tokens
    (31, 128, 30, 2, True),        # F not in quads: element-wise stores
    (33, 192, 36, 3, False),       # an odd number of stages, no bias
    (77, 768, 1000, 2, True),      # three token groups, a ragged last block
    (128, 256, 16640, 1, True),    # 64 features per block
    (129, 256, 4100, 2, True),     # two blocks along the tokens
    (255, 320, 2056, 1, True),
])
def test_short_batches(T, d, F, L, bias, dtype):
    torch.manual_seed(T + d + F)
    x = torch.randn(L, T, d, device="cuda").to(dtype)
    w = (torch.randn(L, F, d, device="cuda") / d ** 0.5).to(dtype)
    b = torch.randn(L, F, device="cuda").to(dtype) if bias else None
    if b is not None and b.stride(0) % 8:        # (any stride is taken)
        b = b.contiguous()
    got = engine.encode(x, w, b)
    ref = torch.bmm(x.double(), w.double().transpose(1, 2).contiguous())
    mag = torch.bmm(x.double().abs(), w.double().abs().transpose(1, 2).contiguous())
    if b is not None:
        ref += b.double()[:, None]
        mag += b.double().abs()[:, None]
    # one rounding of the result plus fp32 sums of d products in any order
    bound = ROUND[dtype] * ref.abs() + (d + 8) * 2.0 ** -24 * mag + (2.0 ** -24 if dtype == torch.float16 else 0.0)
    assert got.shape == ref.shape and bool(((got.double() - ref).abs() <= bound).all())


def test_short_batch_inside_a_larger_output():
    """Layers of the output further apart than their rows: nothing beyond them is written."""
    x, w = torch.randn(2, 40, 128, device="cuda"), torch.randn(2, 50, 128, device="cuda")
    room = torch.full((2, 48, 50), 7.0, device="cuda")
    engine.encode(x, w, None, out=room[:, :40])
    ref = torch.bmm(x.double(), w.double().transpose(1, 2).contiguous())
    assert (room[:, :40].double() - ref).abs().max() < 1e-4 and bool((room[:, 40:] == 7.0).all())
