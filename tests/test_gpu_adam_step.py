"""The Adam step four elements at a time (k_adam_vec) gives the bits of the one for any length and alignment (k_adam)."""
import pytest
import torch

from crosslayer_coding_amd import _native as nat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [4, 1024, 1028, 4 * 256 * 256 * 64 + 4])
def test_quads_and_elements(n, dtype):
    lib, dev = nat.load(), torch.device("cuda:0")
    torch.manual_seed(n % 1000)
    p, g, m = torch.randn(n, device=dev).to(dtype), torch.randn(n, device=dev), torch.randn(n, device=dev)
    v = torch.rand(n, device=dev)
    outs = []
    for shift in (0, 1):                  # one element off a 16-byte boundary: element by element
        ts = []
        for t in (p, g, m, v):
            room = torch.empty(n + 8, dtype=t.dtype, device=dev)
            room[shift:shift + n] = t
            ts.append(room[shift:shift + n])
        nat.check(lib.clt_adam_step(*(nat.ptr(t) for t in ts), n, 1e-2, 0.9, 0.999, 1e-8, 3, nat.dtype_code(dtype),
                                    nat.current_stream(dev)), "clt_adam_step")
        outs.append(ts)
    for a, b in zip(*outs):
        assert torch.equal(a, b)
