"""Which kernel a float32 optimiser step gives the decoders, batch after batch: the kernels stand still, the rule is what runs."""
from types import SimpleNamespace

import pytest
import torch

from crosslayer_coding_amd import engine, optim

L, F, D = 4, 512, 64
KERNELS = {"decoder_weight_grad_adam_tiled": "C", "decoder_grad_adam_rows": "R", "decoder_weight_grad_adam": "S"}


def _steps(monkeypatch, wanted, regroup=None):
    """The routes of a batch for each letter of `wanted`, the fastest by shape (C column tiles, R LDS tiles, S row by row), and how often
    the weights were tiled."""
    took, tiled = [], []
    for name, letter in KERNELS.items():
        monkeypatch.setattr(engine, name, lambda *a, _l=letter, **kw: took.append(_l))
    monkeypatch.setattr(engine, "tile_decoders", lambda packed, d, out=None: tiled.append(1) or torch.empty(1))
    monkeypatch.setattr(engine, "untile_decoders", lambda *a: None)
    monkeypatch.setattr(engine, "decoder_tile_width", lambda *a: 8)
    monkeypatch.setattr(engine, "grad_rows_wanted", lambda T, *a: "CRS".index(wanted[T]))
    n_dec = L * (L + 1) // 2
    weights = [SimpleNamespace(weight=torch.nn.Parameter(torch.zeros(D, F))) for _ in range(n_dec)]
    dec = SimpleNamespace(packed=lambda p=torch.zeros(n_dec, F, D): p, packed_generation=lambda: (1, 0), _ordered=lambda: weights,
                          mark_parameters_behind=lambda: None, skip_weights=None, feature_offset=None, feature_scale=None)
    config = SimpleNamespace(num_layers=L, num_features=F, d_model=D, decoder_tying="none", activation_fn="batchtopk")
    opt = optim.CLTAdam(SimpleNamespace(config=config, device="cpu", decoder_module=dec, _workspace=lambda: None))
    for m in opt.state["dec_w"]:
        m.normal_()
    before = [m.clone() for m in opt.state["dec_w"]]
    if regroup is not None:
        monkeypatch.setattr(opt, "_decoder_moments_to", regroup(opt._decoder_moments_to))
    for T in range(len(wanted)):
        opt.decoder_weight_step(None, SimpleNamespace(T=T, L=L, F=F, capacity=1), torch.zeros(1))
    assert all(torch.equal(a, b) for a, b in zip(before, opt.decoder_moments()))       # regrouped, never changed
    return "".join(took), len(tiled)


@pytest.mark.parametrize("wanted,took,tiled", [
    ("RRSRS", "RRSRS", 0),                     # from rows of moments every batch goes where it is fastest
    ("CRCRCR", "CCCCCC", 1),                   # one batch among others does not put the tiled weights out of date
    ("CRRRC", "CCRRC", 2),                     # a run of them does, from the second one on
    ("CSCSC", "CCCCC", 1),
    ("CSSSSSSSSSC", "CCCCCCCCSSC", 2),         # short lists leave the tiles when they go on
    ("CRRSC", "CCRCC", 2),                     # behind LDS tiles the moments still are in tiles
    ("CSSSSSSSRS", "CCCCCCCCRS", 1),           # nine that were faster elsewhere
])
def test_a_batch_among_others_stays_with_the_tiles(monkeypatch, wanted, took, tiled):
    assert _steps(monkeypatch, wanted) == (took, tiled)


def test_no_room_to_regroup_the_moments(monkeypatch):
    def regroup(real):
        def to(layout, cols=0):
            if layout == "rows":
                raise torch.OutOfMemoryError("no room")
            real(layout, cols)
        return to
    assert _steps(monkeypatch, "C" + "S" * 18, regroup) == ("C" * 19, 3)
