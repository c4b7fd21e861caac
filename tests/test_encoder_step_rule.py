"""Which training steps take the encoder weights' Adam step in the gradient kernel: the ones where it was measured no slower than
gradient and step apart."""
from types import SimpleNamespace

import pytest
import torch

from crosslayer_coding_amd import engine, optim

# tokens, features, survivors per token, widths: us of the two calls / in place, three layers each
SHORT = [(1024, 8192, 24, (116, 91)), (2048, 8192, 64, (155, 144)), (4096, 24576, 200, (607, 521)), (8192, 24576, 200, (1181, 1064))]
LONG = [(4096, 8192, 133, (331, 347)), (4096, 8192, 266, (561, 608)), (8192, 8192, 266, (1314, 1391)), (8192, 24576, 400, (3692, 4004))]


@pytest.mark.parametrize("T,F,k,us", SHORT + LONG)
def test_long_lists_keep_the_two_calls(T, F, k, us):
    assert engine.encoder_step_wanted(3 * T * k, F, 3) == (us[1] <= us[0])


def test_a_step_of_ones_own_sees_the_encoder_gradients():
    class Watching(optim.CLTAdam):
        def step(self, raw):
            self.norm = raw["enc_w"].norm()
            super().step(raw)

    def fuses(cls, patch=False):
        opt = cls.__new__(cls)
        opt.fuse_encoder_step, w = True, torch.zeros(2, 64, 8)
        opt.state = {"enc_w": (w, w)}
        opt.model = SimpleNamespace(encoder_module=SimpleNamespace(stacked=lambda: (w, None)))
        if patch:
            opt.step = lambda raw: None
        return opt.fuses_encoder_step(torch.zeros(2, 16, 8), 128)
    assert fuses(optim.CLTAdam) and not fuses(Watching) and not fuses(optim.CLTAdam, patch=True)
