"""Which training steps take the encoder weights' Adam step in the gradient kernel: the ones where it was measured no slower than
gradient and step apart."""
import pytest

from crosslayer_coding_amd import engine

# tokens, features, survivors per token, widths: us of the two calls / in place, three layers each
SHORT = [(1024, 8192, 24, (116, 91)), (2048, 8192, 64, (155, 144)), (4096, 24576, 200, (607, 521)), (8192, 24576, 200, (1181, 1064))]
LONG = [(4096, 8192, 133, (331, 347)), (4096, 8192, 266, (561, 608)), (8192, 8192, 266, (1314, 1391)), (8192, 24576, 400, (3692, 4004))]


@pytest.mark.parametrize("T,F,k,us", SHORT + LONG)
def test_long_lists_keep_the_two_calls(T, F, k, us):
    assert engine.encoder_step_wanted(3 * T * k, F, 3) == (us[1] <= us[0])
