"""The matrix-core decode (clt_decode_tiles) against dense products in float64, at the edges of its tiles: 512 features,
16 tokens per group, 16 wavefronts x 4 groups per workgroup, 32 entries per batch, 64 columns."""
import pytest
import torch

import crosslayer_coding_amd as cca
from crosslayer_coding_amd import _native as nat
from crosslayer_coding_amd import engine

pytestmark = pytest.mark.gpu


def _lists(L, T, F, per_token, dtype, seed, heavy):
    g = torch.Generator().manual_seed(seed)
    act = torch.zeros(L, T, F)
    for s in range(L):
        keep = torch.rand(T, F, generator=g) < per_token / F
        if heavy:                      # one token with every feature, one source with next to none
            keep[T // 2] = True
            keep[:, F // 2:] &= s != 1
        act[s] = torch.where(keep, torch.randn(T, F, generator=g), torch.zeros(()))
    act = act.to(dtype)
    nz = act.reshape(L * T, F) != 0
    row_ptr = torch.zeros(L * T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(nz.sum(1), 0)
    col = nz.nonzero()[:, 1].int()
    return act, row_ptr, col, act.reshape(L * T, F)[nz]


def _slot(tying, s, t, L):
    return s if tying == "per_source" else s * L - (s * (s - 1)) // 2 + (t - s)


def _run(dev, act, row_ptr, col, val, w, tying, d, bias, skip, t0, t1, mask, f32, cap, guarded):
    L, T, F = act.shape
    lib = nat.load()
    slab = engine.alloc_packed(w.shape[0], F, d, act.dtype, dev)
    slab[:, :, :d] = w.to(dev)
    rp, c, v = row_ptr.to(dev), torch.cat([col, col.new_zeros(1)]).to(dev), torch.cat([val, val.new_zeros(1)]).to(dev)
    b, k = (None if x is None else x.to(dev) for x in (bias, skip))
    out = torch.full((L, T, d), 7.0, dtype=torch.float32 if f32 else act.dtype, device=dev)
    nbytes = lib.clt_decode_tiles_workspace_bytes(T, d, F, L, t1 - t0, cap)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=dev)      # what lies behind the records must not matter
    args = (nat.ptr(rp), nat.ptr(c), nat.ptr(v), nat.ptr(slab), nat.ptr(b), nat.ptr(k), nat.ptr(out), T, d, F, L, nat.TYING[tying],
            t0, t1, mask, nat.dtype_code(act.dtype), 1 if f32 else 0, cap)
    for _ in range(2):                 # the second pass meets a workspace in use
        nat.check(lib.clt_decode_tiles(*args, nat.ptr(ws), ws.numel(), nat.current_stream(rp.device)), "clt_decode_tiles")
        if guarded:
            nat.check(lib.clt_decode_sparse_if_over(*args, nat.current_stream(rp.device)), "clt_decode_sparse_if_over")
    return out.cpu()


@pytest.mark.parametrize("L,T,F,d,per_token,dtype,tying,heavy", [
    (1, 1, 8, 64, 3, torch.bfloat16, "none", False),             # less than one of everything
    (2, 16, 512, 64, 32, torch.bfloat16, "none", False),         # exactly one group, one tile
    (3, 17, 513, 128, 60, torch.float16, "none", False),         # one token and one feature over
    (3, 15, 1024, 64, 200, torch.bfloat16, "per_source", True),
    (2, 1025, 1300, 192, 20, torch.bfloat16, "none", False),     # a workgroup's tokens and one more
    (4, 300, 4096, 64, 1, torch.float16, "none", True),          # most batches empty
    (2, 2100, 640, 256, 40, torch.bfloat16, "per_source", False),
    (3, 64, 2048, 320, 700, torch.bfloat16, "none", True),       # far denser than the kernel is meant for
])
def test_decode_tiles_against_dense_products(L, T, F, d, per_token, dtype, tying, heavy):
    dev = torch.device("cuda:0")
    act, row_ptr, col, val = _lists(L, T, F, per_token, dtype, seed=L * 1000 + T, heavy=heavy)
    g = torch.Generator().manual_seed(5)
    n_dec = L if tying == "per_source" else L * (L + 1) // 2
    w = (torch.rand(n_dec, F, d, generator=g) - 0.5).to(dtype)
    bias, skip = torch.randn(L, d, generator=g), torch.randn(L, T, d, generator=g)
    full = (1 << L) - 1
    cases = [(0, L, full, True, None, None), (0, L, full, False, bias, skip)]
    if L > 2:
        cases.append((1, L, full & ~2, True, bias, None))        # a layer left out although it has survivors
    for t0, t1, mask, f32, b, k in cases:
        got = _run(dev, act, row_ptr, col, val, w, tying, d, b, k, t0, t1, mask, f32, col.numel(), False)
        for t in range(L):
            if not t0 <= t < t1:
                assert (got[t] == 7.0).all()
                continue
            ref, mag, n = torch.zeros(T, d, dtype=torch.float64), torch.zeros(T, d, dtype=torch.float64), torch.zeros(T, 1)
            for s in range(t + 1):
                if mask >> s & 1:
                    a, m = act[s].double(), w[_slot(tying, s, t, L)].double()
                    ref += a @ m
                    mag += a.abs() @ m.abs()
                    n += (act[s] != 0).sum(1, keepdim=True)
            for extra in (None if b is None else b[t].double(), None if k is None else k[t].double()):
                if extra is not None:
                    ref, mag = ref + extra, mag + extra.abs()
            # products of two 16-bit numbers are exact in fp32; each of the n + 2 additions is off by at most 2^-23 of what
            # has been summed, and the result is rounded once to the output type
            bound = (n.double() + 2) * 2.0 ** -23 * mag
            if not f32:
                bound = bound + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * (ref.abs() + bound) + 2.0 ** -24
            assert (got[t].double() - ref).abs().le(bound).all(), (t, (got[t].double() - ref).abs().max())


@pytest.mark.parametrize("pattern", ["one class", "every column", "two entries", "33 entries", "one row of a group"])
def test_decode_tiles_wherever_entries_are_dealt_to(pattern):
    """Tiles whose entries fall into one class of columns (all half reads of a batch meet it), fill more batches than a
    wavefront puts together at a time, or leave most places of a batch empty."""
    dev = torch.device("cuda:0")
    L, T, F, d = 1, 40, 1100, 64
    g = torch.Generator().manual_seed(11)
    act = torch.randn(L, T, F, generator=g).bfloat16()
    cols, rows = torch.arange(F), torch.arange(T).unsqueeze(1)
    keep = {"one class": (cols % 8 == 3) & (rows >= 0), "every column": (cols >= 0) & (rows >= 0),
            "two entries": (cols % 512 == 17) & (rows % 16 < 2), "33 entries": (cols % 512 < 11) & (rows % 16 < 3),
            "one row of a group": (cols % 3 == 0) & (rows % 16 == 5)}[pattern]
    act[0][~keep] = 0
    nz = act.reshape(T, F) != 0
    row_ptr = torch.zeros(T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(nz.sum(1), 0)
    col, val = nz.nonzero()[:, 1].int(), act.reshape(T, F)[nz]
    w = (torch.rand(1, F, d, generator=g) - 0.5).bfloat16()
    got = _run(dev, act, row_ptr, col, val, w, "none", d, None, None, 0, 1, 1, True, col.numel(), False)
    ref, mag = act[0].double() @ w[0].double(), act[0].double().abs() @ w[0].double().abs()
    # exact products; each addition is off by at most 2^-23 of what has been summed
    assert (got[0].double() - ref).abs().le((nz.sum(1, keepdim=True).double() + 2) * 2.0 ** -23 * mag).all()


def test_decode_tiles_of_empty_lists():
    """No stream has a record: every wavefront meets the one behind the last stream."""
    dev = torch.device("cuda:0")
    L, T, F, d = 2, 40, 1100, 128
    act, row_ptr, col, val = _lists(L, T, F, 0, torch.bfloat16, seed=3, heavy=False)
    w = (torch.rand(3, F, d, generator=torch.Generator().manual_seed(1)) - 0.5).bfloat16()
    bias = torch.randn(L, d, generator=torch.Generator().manual_seed(2))
    for cap in (0, 1000):
        got = _run(dev, act, row_ptr, col, val, w, "none", d, bias, None, 0, L, 3, True, cap, False)
        assert torch.equal(got, bias.unsqueeze(1).expand(L, T, d))


def test_decode_tiles_leaves_longer_lists_to_the_gather():
    dev = torch.device("cuda:0")
    L, T, F, d = 2, 100, 1000, 128
    act, row_ptr, col, val = _lists(L, T, F, 30, torch.bfloat16, seed=3, heavy=False)
    w = (torch.rand(3, F, d, generator=torch.Generator().manual_seed(1)) - 0.5).bfloat16()
    n = col.numel()
    exact = _run(dev, act, row_ptr, col, val, w, "none", d, None, None, 0, L, 3, True, n, True)
    over = _run(dev, act, row_ptr, col, val, w, "none", d, None, None, 0, L, 3, True, n - 1, True)
    left = _run(dev, act, row_ptr, col, val, w, "none", d, None, None, 0, L, 3, True, n - 1, False)
    assert (left == 7.0).all()
    assert torch.allclose(exact, over, rtol=0, atol=60 * 2.0 ** -23 * 60)      # 60 terms below 60 in sum, summed in another order


@pytest.mark.parametrize("L,T,F,d,per_token,dtype,tying,heavy", [
    (1, 1, 8, 64, 3, torch.bfloat16, "none", False),
    (3, 17, 513, 192, 60, torch.float16, "none", False),
    (5, 130, 1100, 704, 90, torch.bfloat16, "per_source", True),           # units that are no whole rounds over the XCDs
    (2, 40, 70000, 64, 900, torch.bfloat16, "none", False),                # indices of more than 16 bits
    (3, 1900, 1024, 1024, 3, torch.float16, "none", False),                # more blocks than workgroups
    (64, 3, 600, 64, 4, torch.bfloat16, "per_source", False),
])
def test_gather_of_longer_lists(L, T, F, d, per_token, dtype, tying, heavy):
    """clt_decode_sparse_if_over in place of the tiles that leave such a list alone, against dense products."""
    dev = torch.device("cuda:0")
    act, row_ptr, col, val = _lists(L, T, F, per_token, dtype, seed=L + T, heavy=heavy)
    g = torch.Generator().manual_seed(5)
    n_dec = L if tying == "per_source" else L * (L + 1) // 2
    w = (torch.rand(n_dec, F, d, generator=g) - 0.5).to(dtype)
    bias, skip = torch.randn(L, d, generator=g), torch.randn(L, T, d, generator=g)
    full, n = (1 << L) - 1, col.numel()
    for t0, t1, mask, f32, b, k in [(0, L, full, True, None, None), (L // 2, L, full & ~2, False, bias, skip)]:
        got = _run(dev, act, row_ptr, col, val, w, tying, d, b, k, t0, t1, mask, f32, n - 1, True)
        for t in range(L):
            if not t0 <= t < t1:
                assert (got[t] == 7.0).all()
                continue
            ref, mag, cnt = torch.zeros(T, d, dtype=torch.float64), torch.zeros(T, d, dtype=torch.float64), torch.zeros(T, 1)
            for s in range(t + 1):
                if mask >> s & 1:
                    a, m = act[s].double(), w[_slot(tying, s, t, L)].double()
                    ref, mag, cnt = ref + a @ m, mag + a.abs() @ m.abs(), cnt + (act[s] != 0).sum(1, keepdim=True)
            for extra in (None if b is None else b[t].double(), None if k is None else k[t].double()):
                if extra is not None:
                    ref, mag = ref + extra, mag + extra.abs()
            # as above; the eight lane groups' sums meet in three more additions
            bound = (cnt.double() + 6) * 2.0 ** -23 * mag
            if not f32:
                bound = bound + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * (ref.abs() + bound) + 2.0 ** -24
            assert (got[t].double() - ref).abs().le(bound).all(), (t, (got[t].double() - ref).abs().max())


def test_a_captured_decode_follows_a_threshold_list_that_outgrows_its_estimate(monkeypatch):
    """The room is fixed when the graph is captured; replays on thin and dense lists, with eager work between them."""
    dev = torch.device("cuda:0")
    L, T, F, d = 3, 600, 4096, 128
    monkeypatch.setattr(nat.load(), "clt_decode_tiles_wanted", lambda *a: 1)
    lists = {k: _lists(L, T, F, k, torch.bfloat16, seed=k, heavy=False) for k in (10, 100)}
    assert lists[10][2].numel() < 20000 < 2 * 20000 + 65536 < lists[100][2].numel()
    cap = lists[100][2].numel() + 1000
    surv = engine.SurvivorList(torch.zeros(L * T + 1, dtype=torch.int32, device=dev), torch.zeros(cap, dtype=torch.int32, device=dev),
                               torch.zeros(cap, dtype=torch.bfloat16, device=dev), T, F, L, torch.bfloat16,
                               torch.zeros(1, dtype=torch.int32, device=dev), 20000)
    w = engine.alloc_packed(L * (L + 1) // 2, F, d, torch.bfloat16, dev)
    w[:, :, :d] = torch.randn(L * (L + 1) // 2, F, d, generator=torch.Generator().manual_seed(1)).bfloat16().to(dev)
    ws = engine.Workspace(dev)

    def fill(k):
        _, row_ptr, col, val = lists[k]
        surv.row_ptr.copy_(row_ptr)
        surv.col[: col.numel()].copy_(col)
        surv.val[: val.numel()].copy_(val)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fill(10)
        engine.decode_sparse(surv, w, "none", d, ws=ws)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = engine.decode_sparse(surv, w, "none", d, ws=ws)
    for k in (100, 10, 100, 100, 10):
        fill(k)
        graph.replay()
        got = out.float()
        eager = engine.decode_sparse(surv, w, "none", d, ws=ws).float()
        ref = engine.decode_sparse(surv, w, "none", d, ws=None).float()
        torch.cuda.synchronize()
        assert torch.equal(got, eager)
        # the same sums in another order, rounded to bf16: a last place where that decides
        assert bool(((got - ref).abs() <= 2.0 ** -7 * ref.abs() + 1e-3).all()) and float(ref.norm()) > 0


def test_a_denser_eager_batch_leaves_the_captured_graph_its_room(monkeypatch):
    """The room of a threshold list follows the last total seen, so an eager batch of the captured shape can outgrow the buffer
    that the graph writes: memory allocated afterwards must not be that buffer's."""
    dev = torch.device("cuda:0")
    L, T, F, d = 3, 600, 4096, 128
    monkeypatch.setattr(nat.load(), "clt_decode_tiles_wanted", lambda *a: 1)
    _, row_ptr, col, val = _lists(L, T, F, 10, torch.bfloat16, seed=3, heavy=False)
    surv = engine.SurvivorList(row_ptr.to(dev), col.to(dev), val.to(dev), T, F, L, torch.bfloat16,
                               torch.zeros(1, dtype=torch.int32, device=dev), 20000)
    w = engine.alloc_packed(L * (L + 1) // 2, F, d, torch.bfloat16, dev)
    w[:, :, :d] = torch.randn(L * (L + 1) // 2, F, d, generator=torch.Generator().manual_seed(1)).bfloat16().to(dev)
    ws = engine.Workspace(dev)
    monkeypatch.setattr(engine.SurvivorList, "capacity", 1 << 30)      # arrays for any list the shape can produce
    want = engine.decode_sparse(surv, w, "none", d, ws=ws)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = engine.decode_sparse(surv, w, "none", d, ws=ws)
    room = ws.get("decode_tiles", 0).numel()
    surv.nnz_hint = 200000
    assert torch.equal(engine.decode_sparse(surv, w, "none", d, ws=ws), want)
    assert ws.get("decode_tiles", 0).numel() > room
    later = [torch.full((room,), 7, dtype=torch.uint8, device=dev) for _ in range(4)]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and all(bool((t == 7).all()) for t in later)


def test_an_outgrown_threshold_list_costs_what_the_gather_costs():
    """Rows of more than five registers' worth of pieces, for which a single pass over the sources has only the kernel for any
    shape (28 times the gather's time here); the gather measured beside it, the best of five, allowed a factor of four."""
    dev = torch.device("cuda:0")
    L, T, F, d, k = 4, 512, 8192, 2560, 50
    g = torch.Generator(device=dev).manual_seed(1)
    rows, n = L * T, L * T * k
    col = (torch.rand(rows, k, generator=g, device=dev) * (F // k)).int() + torch.arange(k, device=dev, dtype=torch.int32) * (F // k)
    ptr = torch.arange(0, n + 1, k, dtype=torch.int32, device=dev)
    val = torch.randn(n, generator=g, device=dev).bfloat16()
    w = engine.alloc_packed(L * (L + 1) // 2, F, d, torch.bfloat16, dev)
    w[:, :, :d] = torch.randn(F, d, generator=g, device=dev).bfloat16()
    ws, lib, stream = engine.Workspace(dev), nat.load(), nat.current_stream(dev)
    out, over = (torch.empty(L, T, d, dtype=torch.bfloat16, device=dev) for _ in range(2))
    wbuf = ws.get("decode", lib.clt_decode_workspace_bytes(T, d, F, L))
    shape = (T, d, F, L, nat.TYING["none"], 0, L, (1 << L) - 1, nat.CLT_BF16, 0)
    head = (nat.ptr(ptr), nat.ptr(col), nat.ptr(val), nat.ptr(w))
    calls = {"gather": lambda: lib.clt_decode_sparse(*head, None, None, None, None, nat.ptr(out), *shape, nat.ptr(wbuf), wbuf.numel(), stream),
             "over": lambda: lib.clt_decode_sparse_if_over(*head, None, None, nat.ptr(over), *shape, n - 1, stream)}
    ms = {}
    for name, call in calls.items():
        best = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            assert call() == 0
            b.record()
            torch.cuda.synchronize()
            best.append(a.elapsed_time(b))
        ms[name] = min(best[1:])
    assert float((out.float() - over.float()).norm() / out.float().norm()) < 1e-3      # bf16 results of sums in another order
    assert ms["over"] <= 4 * ms["gather"], ms


def test_decode_tiles_keeps_tokens_apart():
    """Values that are not finite stay with their token although sixteen tokens share every product."""
    dev = torch.device("cuda:0")
    L, T, F, d = 1, 32, 512, 64
    act, row_ptr, col, val = _lists(L, T, F, 40, torch.bfloat16, seed=9, heavy=False)
    w = (torch.rand(1, F, d, generator=torch.Generator().manual_seed(1)) + 0.5).bfloat16()
    val = val.clone()
    val[row_ptr[3]] = float("nan")
    val[row_ptr[7]] = float("inf")
    got = _run(dev, act, row_ptr, col, val, w, "none", d, None, None, 0, 1, 1, True, col.numel(), False)[0]
    fine = torch.ones(T, dtype=torch.bool)
    fine[[3, 7]] = False
    assert got[3].isnan().all() and (got[7] == float("inf")).all() and got[fine].isfinite().all()


def test_the_model_takes_the_tiles_when_they_are_priced_lower():
    lib = nat.load()
    want = lambda T, k, **kw: lib.clt_decode_tiles_wanted(T, 768, 24576, 12, 12, 12 * T * k, nat.TYING[kw.get("tying", "none")],  # noqa: E731
                                                          nat.dtype_code(kw.get("dtype", torch.bfloat16)))
    assert want(4096, 200) == 1 and want(4096, 200, tying="per_source") == 1 and want(4096, 200, dtype=torch.float16) == 1
    assert want(64, 200) == 0 and want(4096, 2) == 0
    assert want(4096, 200, dtype=torch.float32) == 0 and want(4096, 200, tying="per_target") == 0
    assert cca is not None


@pytest.mark.parametrize("entries", [256, 257, 288, 511, 2049, 8192])
def test_decode_tiles_of_tiles_with_many_entries(entries):
    """A tile of 16 tokens x 512 features with as many entries as are put together in LDS, one more, whole batches, all."""
    dev = torch.device("cuda:0")
    L, T, F, d = 1, 33, 1024, 64
    g = torch.Generator().manual_seed(entries)
    act = torch.randn(L, T, F, generator=g).bfloat16()
    act[act == 0] = 1.0
    keep = torch.rand(T, F, generator=g) < 0.02
    tile = torch.zeros(16 * 512, dtype=torch.bool)
    tile[torch.randperm(16 * 512, generator=g)[:entries]] = True
    keep[16:32, 512:] = tile.view(16, 512)
    act[0][~keep] = 0
    row_ptr = torch.zeros(T + 1, dtype=torch.int32)
    row_ptr[1:] = torch.cumsum(keep.sum(1), 0)
    col, val = keep.nonzero()[:, 1].int(), act[0][keep]
    w = (torch.rand(1, F, d, generator=g) - 0.5).bfloat16()
    got = [_run(dev, act, row_ptr, col, val, w, "none", d, None, None, 0, 1, 1, True, col.numel(), False) for _ in range(2)]
    assert torch.equal(got[0], got[1])
    ref, mag = act[0].double() @ w[0].double(), act[0].double().abs() @ w[0].double().abs()
    # exact products; each addition is off by at most 2^-23 of what has been summed
    assert (got[0][0].double() - ref).abs().le((keep.sum(1, keepdim=True).double() + 2) * 2.0 ** -23 * mag).all()
