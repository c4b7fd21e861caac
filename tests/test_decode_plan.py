"""Which decode a survivor list is handed to, checked without a GPU: tensors without storage, native launches recorded in place
of made."""
import weakref

import pytest
import torch

from crosslayer_coding_amd import _native as nat
from crosslayer_coding_amd import engine


class _Recorder:
    """The native library with its decode launches recorded.  Their argument checks run: a workspace of no bytes is the last
    thing they refuse, before anything is launched."""

    def __init__(self, lib):
        self._lib, self.calls = lib, []

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def clt_decode_tiles(self, *args):
        self.calls.append(("tiles", args))
        code = self._lib.clt_decode_tiles(*args[:-2], 0, args[-1])
        return 0 if code == -3 else code      # CLT_ERR_WORKSPACE

    def clt_decode_sparse_if_over(self, *args):
        self.calls.append(("if_over", args))
        return 0

    def clt_decode_sparse(self, *args):
        self.calls.append(("gather", args))
        return 0


@pytest.fixture
def recorder(monkeypatch):
    rec = _Recorder(nat.load())
    monkeypatch.setattr(nat, "load", lambda *a, **k: rec)
    monkeypatch.setattr(nat, "require_device", lambda *a: None)
    monkeypatch.setattr(nat, "ptr", lambda t: None if t is None else 4096)
    monkeypatch.setattr(engine, "_stream", lambda t: None)
    return rec


def _decode(L, T, d, F, hint, dtype=torch.bfloat16, **kw):
    meta = torch.device("meta")
    cap = engine.max_list_entries(L, T, F)
    surv = engine.SurvivorList(torch.empty(L * T + 1, dtype=torch.int32, device=meta), torch.empty(cap, dtype=torch.int32, device=meta),
                               torch.empty(cap, dtype=dtype, device=meta), T, F, L, dtype,
                               torch.empty(1, dtype=torch.int32, device=meta), hint)
    w = torch.empty((L * (L + 1) // 2, F, engine.decoder_pitch(d, dtype)), dtype=dtype, device=meta)
    return engine.decode_sparse(surv, w, "none", d, ws=engine.Workspace(meta), **kw)


@pytest.mark.parametrize("L,d,F,T,density", [
    (24, 1024, 32768, 29000, None),         # the first forward of a threshold model: 1 % of the features assumed
    (24, 1024, 32768, 29000, 0.01), (24, 1024, 32768, 43500, 0.006), (12, 768, 49152, 57500, 0.006),
    (12, 768, 24576, 4096, 0.008), (12, 768, 24576, 65536, 0.008),
])
def test_a_threshold_list_of_a_long_batch_is_decoded(recorder, L, d, F, T, density):
    """The records can count fewer survivors than twice the estimate of such a batch: room for as many as they can."""
    hint = None if density is None else int(L * T * F * density)
    _decode(L, T, d, F, hint)
    names = [name for name, _ in recorder.calls]
    assert names in (["tiles", "if_over"], ["gather"])
    if names[0] == "tiles":
        cap = recorder.calls[0][1][17]
        assert cap == recorder.calls[1][1][17] and (hint or L * T * F // 100) <= cap
        assert cap <= recorder.clt_decode_tiles_max_entries(T, d, F, L, L)


def test_max_entries_is_the_largest_that_is_taken(recorder):
    for L, T, d, F in ((24, 30000, 1024, 32768), (1, 1, 64, 8), (12, 4096, 768, 24576)):
        n = recorder.clt_decode_tiles_max_entries(T, d, F, L, L)
        args = (4096, 4096, 4096, 4096, None, None, 4096, T, d, F, L, 0, 0, L, 1, nat.CLT_BF16, 0)
        assert recorder._lib.clt_decode_tiles(*args, n, 4096, 0, None) == -3            # CLT_ERR_WORKSPACE
        assert recorder._lib.clt_decode_tiles(*args, n + 1, 4096, 0, None) == -6        # CLT_ERR_RANGE
    assert recorder.clt_decode_tiles_max_entries(4096, 768, 513 * 512, 12, 12) == 0     # more tiles than the kernels take


def test_a_buffer_that_a_captured_graph_writes_outlives_its_successor(monkeypatch):
    """A denser batch of the captured shape outgrows the room of a threshold list; the graph's replays go on writing the old one."""
    ws = engine.Workspace(torch.device("cpu"))
    capturing = False
    monkeypatch.setattr(engine, "_capturing", lambda device: capturing, raising=False)
    alive = []
    for grown_by, held in ((1, 0), (2, 1), (3, 1)):      # before a capture, right after one, once more
        capturing = grown_by == 2
        old = ws.get("list", 1000 * grown_by)
        capturing = False
        alive.append(weakref.ref(old))
        del old
        ws.get("list", 1000 * (grown_by + 1))
        assert sum(r() is not None for r in alive) == held
    ws.release()
    assert all(r() is None for r in alive)


class _ThinRecorder(_Recorder):
    def clt_decode_thin_wanted(self, *args):
        return 1

    def clt_decode_thin(self, *args):
        self.calls.append(("thin", args))
        return 0

    def clt_decode_thin_up_to(self, *args):
        self.calls.append(("thin_up_to", args))
        return 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hint", [None, 180000])
@pytest.mark.parametrize("exact", [True, False])
def test_an_estimated_total_is_checked_on_the_device(recorder, monkeypatch, dtype, hint, exact):
    """The gather for thin lists takes a list whose length is known; one whose length is estimated only where another
    decode stands by for what the estimate left out."""
    rec = _ThinRecorder(recorder._lib)
    monkeypatch.setattr(nat, "load", lambda *a, **k: rec)
    L, T, d, F, meta = 12, 3000, 768, 24576, torch.device("meta")
    cap = 600000 if exact else engine.max_list_entries(L, T, F)
    surv = engine.SurvivorList(torch.empty(L * T + 1, dtype=torch.int32, device=meta), torch.empty(cap, dtype=torch.int32, device=meta),
                               torch.empty(cap, dtype=dtype, device=meta), T, F, L, dtype,
                               None if exact else torch.empty(1, dtype=torch.int32, device=meta), hint, True)
    w = torch.empty((L * (L + 1) // 2, F, engine.decoder_pitch(d, dtype)), dtype=dtype, device=meta)
    engine.decode_sparse(surv, w, "none", d, ws=engine.Workspace(meta))
    names = [name for name, _ in rec.calls]
    if exact:
        assert names == ["thin"]
    elif dtype == torch.float32:
        assert names == ["gather"]
    else:
        assert names == ["thin_up_to", "if_over"]
        assert rec.calls[0][1][17] == rec.calls[1][1][17] >= (hint or L * T * F // 100)


@pytest.mark.parametrize("dtype,widths", [(torch.bfloat16, (512, 768, 1024, 2048)), (torch.float16, (512, 768, 1024, 2048)),
                                          (torch.float32, (512, 768, 1024))])
def test_widths_of_the_gather_for_thin_lists(dtype, widths):
    """Others are refused by the decode and never wanted by its rule."""
    lib, code = nat.load(), nat.dtype_code(dtype)
    for d in (64, 128, 256, 512, 640, 768, 1000, 1024, 1280, 1536, 1792, 2048, 2304, 4096):
        assert lib.clt_decode_thin_wanted(3000, d, 24576, 12, 12, 100000, 0, code) == (1 if d in widths else 0), d
        # (widths that are taken get as far as the check of the addresses: CLT_ERR_ALIGN)
        got = lib.clt_decode_thin(4096, 4096, 4096, 4100, None, None, 4096, 3000, d, 24576, 12, 0, 0, 12, 1, code, 0, None)
        assert (got == -5) == (d in widths) and got < 0, (d, got)
        assert lib.clt_decode_thin_up_to(4096, 4096, 4096, 4100, None, None, 4096, 3000, d, 24576, 12, 0, 0, 12, 1, code, 0, 5, None) == got
