"""The compiled call layer (csrc/host.cpp) against the Python path it stands in
for: the same call with the extension's functions handing everything back gives
the same bits, over the layouts both accept (views, offsets, size-1 dimensions,
padded rows, every table type) and those both copy (misaligned, odd strides), in
the output, the pools and the errors; and the extension takes these calls (one
handed back pays for the refused call and then for all of the Python path)."""

from __future__ import annotations

import math
import types

import pytest
import torch

from engine import _lib
from engine.attention import flash_attention, paged_attention, paged_prefill
from engine.cache import KVCacheConfig, PagedKVCache, kv_append
from engine.model import attention_section, attention_section_rows
from engine.model.rope import build_rope_cache
from engine.quant import int8_matmul

pytestmark = pytest.mark.gpu
DEV = "cuda"
NAMES = ("flash", "paged", "section", "append", "append_seq", "gather", "int8")


def _python_only(m):
    back = types.SimpleNamespace(**{n: (lambda *args: None) for n in NAMES})
    m.setattr(_lib, "host", lambda: back)


def _both(monkeypatch, call, taken=True):
    """call() through the extension and through Python alone: the same tensors,
    or the same refusal (an append of rows with odd strides). taken: the
    extension hands no call back (unless it is refused)."""

    def outcome():
        try:
            return call()
        except ValueError as e:
            return str(e)

    host, back = _lib.host(), []

    def noting(name):
        def f(*args):
            done = getattr(host, name)(*args)
            if done is None:
                back.append(name)
            return done

        return f

    with monkeypatch.context() as m:
        m.setattr(_lib, "host", lambda: types.SimpleNamespace(**{n: noting(n) for n in NAMES}))
        a = outcome()
    assert not (taken and back and not isinstance(a, str)), back
    with monkeypatch.context() as m:
        _python_only(m)
        b = outcome()
    assert type(a) is type(b)
    if isinstance(a, str):
        assert a == b
        return
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype
        assert torch.equal(x.nan_to_num(7.0), y.nan_to_num(7.0)) and torch.equal(x.isnan(), y.isnan())


def _views(g, B, H, L, D, dtype):
    """One (B, H, L, D) tensor in the layouts callers hold."""
    base = torch.randn(B, H, L, D, generator=g).to(dtype).to(DEV)
    padded = torch.empty(B, H, L, D + 8, dtype=dtype, device=DEV)[..., :D]
    padded.copy_(base)
    odd = torch.empty(B, H, L, D + 1, dtype=dtype, device=DEV)[..., :D]
    odd.copy_(base)
    shifted = torch.empty(base.numel() + 1, dtype=dtype, device=DEV)[1:].view(B, H, L, D)
    shifted.copy_(base)
    return [base, base.transpose(1, 2).contiguous().transpose(1, 2), padded, odd, shifted,
            base.transpose(2, 3).contiguous().transpose(2, 3)]


@pytest.mark.parametrize("B,H,Hk,M,N,D", [(1, 4, 2, 5, 700, 64), (2, 2, 1, 130, 130, 128), (1, 1, 1, 1, 1, 32),
                                          (2, 4, 4, 3, 0, 64), (0, 4, 2, 3, 9, 64)])
def test_flash(monkeypatch, B, H, Hk, M, N, D):
    g = torch.Generator().manual_seed(B + M)
    cos, sin = (t.to(DEV) for t in build_rope_cache(2048, D))
    pos = torch.full((B,), 7, dtype=torch.int32, device=DEV)
    for q, k, v in zip(*(_views(g, B, h, n, D, torch.float16) for h, n in ((H, M), (Hk, N), (Hk, N)))):
        for kw in ({}, {"causal": True, "scale": -0.3}, {"rope": (cos, sin)}, {"rope": (cos.half(), sin.half()), "q_pos0": pos},
                   {"causal": 1, "out": torch.empty(B, M, H, D, dtype=torch.float16, device=DEV).transpose(1, 2)}):
            _both(monkeypatch, lambda: (flash_attention(q, k, v, **kw).clone(),))


@pytest.mark.parametrize("L,D,dtype", [(1, 64, torch.float16), (5, 128, torch.bfloat16), (90, 64, torch.float16)])
@pytest.mark.parametrize("rope", [None, "f32", "x"])
def test_sections(monkeypatch, L, D, dtype, rope):
    Hq, Hk, hist = 8, 2, [70, 0, 33, 400]
    g = torch.Generator().manual_seed(L)
    cos, sin = build_rope_cache(1024, D)
    tabs = None if rope is None else tuple(t.to(DEV, torch.float32 if rope == "f32" else dtype) for t in (cos, sin))
    data = [torch.randn(400, 16, Hk, D, generator=g).to(dtype).to(DEV) for _ in range(2)]
    B = len(hist)
    qs, ks, vs = (_views(g, B, h, L, D, dtype) for h in (Hq, Hk, Hk))

    def run(q, k, v, plan, rows):
        cache = PagedKVCache(KVCacheConfig(1, Hk, D, 400, 16, dtype, DEV))
        cache.k[0].copy_(data[0]), cache.v[0].copy_(data[1])
        tables = [cache.new_sequence() for _ in hist]
        for t, n in zip(tables, hist):
            t.length = n
        step = cache.prepare_step(tables, L, num_heads=Hq if plan else None)
        if rows:
            q, k, v = (x.transpose(1, 2).reshape(B * L, -1, D) for x in (q, k, v))
            o = attention_section_rows(q, k, v, 0, cache, step, rope=tabs)
        else:
            o = attention_section(q, k, v, 0, cache, step, rope=tabs)
        return o, cache.k[0], cache.v[0]

    for q, k, v in zip(qs, ks, vs):
        for plan, rows in ((False, False), (True, False), (False, True)):
            _both(monkeypatch, lambda: run(q, k, v, plan, rows))


def test_paged(monkeypatch):
    g = torch.Generator().manual_seed(3)
    kp, vp = (torch.randn(40, 16, 2, 64, generator=g).half().to(DEV) for _ in range(2))
    bt = torch.randperm(40, generator=g).view(2, 20).int().to(DEV)
    lens = torch.tensor([300, 17], dtype=torch.int32, device=DEV)
    for q in _views(g, 2, 4, 3, 64, torch.float16):
        for t, n in ((bt, lens), (bt.long(), lens.long()), (bt.repeat(1, 2)[:, :20], lens)):
            for kw in ({}, {"max_context": 310, "scale": 0.2}, {"causal": False}, {"max_context": 16}):
                _both(monkeypatch, lambda: (paged_attention(q, kp, vp, t, n, **kw), paged_prefill(q, kp, vp, t, n, **kw)))


@pytest.mark.parametrize("M,N,K", [(1, 24, 64), (3, 40, 100), (130, 136, 192), (65, 40, 1000), (0, 8, 64)])
def test_int8(monkeypatch, M, N, K):
    g = torch.Generator().manual_seed(M + K)
    w = torch.randint(-127, 128, (N, K), generator=g).to(torch.int8).to(DEV)
    wp = torch.empty(N, K + 16 - K % 16, dtype=torch.int8, device=DEV)[:, :K]
    wp.copy_(w)
    s = torch.rand(N, generator=g).to(DEV)
    for dtype in (torch.float16, torch.bfloat16):
        x = torch.randn(M, K, generator=g).to(dtype).to(DEV)
        xp = torch.empty(M, K + 8, dtype=dtype, device=DEV)[:, :K]
        xp.copy_(x)
        for xx in (x, xp, x.view(1, M, K), x.t().contiguous().t()):
            for ww in (w, wp):
                for ss in (s, s.half(), s.double()):
                    for b in (None, s.to(dtype), s.half(), torch.nn.Parameter(s), s.repeat(2)[::2]):
                        _both(monkeypatch, lambda: (int8_matmul(xx, ww, ss, bias=b),), taken=M > 0)


def test_errors_keep_their_types():
    q = torch.zeros(1, 2, 4, 64, dtype=torch.float16, device=DEV)
    for bad in (q.float(), q[..., :48], q.cpu()):
        with pytest.raises((ValueError, RuntimeError)):
            flash_attention(bad, bad, bad)
    with pytest.raises(ValueError):
        flash_attention(q, q, q, scale=math.inf)  # refused by the library
    with pytest.raises(ValueError):
        flash_attention(q, q, q, out=torch.empty(1, 2, 4, 65, dtype=torch.float16, device=DEV)[..., :64])
    with pytest.raises(ValueError):
        flash_attention(q, q, q, rope=(torch.zeros(4, 32, device=DEV), torch.zeros(5, 32, device=DEV)))


@pytest.mark.parametrize("Hk,D,bs,dtype", [(8, 64, 16, torch.float16), (2, 128, 5, torch.bfloat16), (3, 16, 1, torch.float16),
                                           (2, 256, 32, torch.bfloat16)])
def test_append_and_gather_of_one_sequence(monkeypatch, Hk, D, bs, dtype):
    """Rows to and from scattered blocks, starts inside a block, and (one-token
    blocks) more block ids than one launch's arguments hold."""
    g = torch.Generator().manual_seed(D + bs)
    N = 1700
    data = [torch.randn(N // bs + 9, bs, Hk, D, generator=g).to(dtype).to(DEV) for _ in range(2)]
    order = torch.randperm(N // bs + 9, generator=g).tolist()

    def run(rows, start, shape):
        cache = PagedKVCache(KVCacheConfig(1, Hk, D, N // bs + 9, bs, dtype, DEV))
        cache.k[0].copy_(data[0]), cache.v[0].copy_(data[1])
        cache._free = list(order)
        t = cache.new_sequence()
        t.blocks = [cache._alloc_block() for _ in range(-(-start // bs))]
        t.length = start
        gg = torch.Generator().manual_seed(rows)
        k, v = (shape(torch.randn(rows, Hk, D, generator=gg).to(dtype).to(DEV)) for _ in range(2))
        cache.append(0, t, k, v)
        assert t.length == start + rows
        return (*cache.gather(0, t), cache.k[0], cache.v[0])

    views = (lambda x: x, lambda x: x.transpose(0, 1).contiguous().transpose(0, 1),
             lambda x: torch.cat([x, x], dim=2)[:, :, :D])
    for rows, start in ((1, 0), (5, 700), (33, 31), (1000, 3), (1, 1600)):
        for shape in views:
            _both(monkeypatch, lambda: run(rows, start, shape))


def test_gather_of_other_caches(monkeypatch):
    """An fp32 cache (gathered, never attended over) and an empty sequence."""
    for dtype, D in ((torch.float32, 24), (torch.float16, 12)):
        cache = PagedKVCache(KVCacheConfig(1, 2, D, 6, 4, dtype, DEV))
        cache.k[0].normal_(), cache.v[0].normal_()
        t = cache.new_sequence()
        assert cache.gather(0, t)[0].shape == (0, 2, D)
        t.blocks, t.length = [5, 0, 3], 10
        _both(monkeypatch, lambda: cache.gather(0, t), taken=dtype == torch.float32)


@pytest.mark.parametrize("rope", [False, True])
def test_append_with_status_and_wide_indices(monkeypatch, rope):
    """kv_append of int64 tables, counts and starts, with a status word of
    either type: the pools and the status (a block id and, with rope, a
    position out of range)."""
    g = torch.Generator().manual_seed(4)
    k, v = (torch.randn(9, 2, 64, generator=g).half().to(DEV) for _ in range(2))
    tabs = tuple(t.to(DEV) for t in build_rope_cache(60, 64)) if rope else None
    bt = torch.tensor([[3, 1, 99, 5], [0, 2, 4, 6]], device=DEV)
    cu, start = torch.tensor([0, 5, 9], device=DEV), torch.tensor([29, 58], device=DEV)

    def run(index, word):
        kp, vp = (torch.zeros(8, 16, 2, 64, dtype=torch.float16, device=DEV) for _ in range(2))
        status = None if word is None else torch.zeros(1, dtype=torch.int32, device=DEV).view(word)
        kv_append(k, v, kp, vp, *(x.to(index) for x in (bt, cu, start)), 5, status, rope=tabs)
        if word is not None:
            assert status.view(torch.int32).item() == (3 if rope else 1)
        return kp, vp

    for index in (torch.int32, torch.int64):
        for word in (None, torch.int32, torch.uint32):
            _both(monkeypatch, lambda: run(index, word))


@pytest.fixture
def no_memory():
    """Nothing over 4 MB can be allocated while it is entered (the caching
    allocator's own limit: the driver is never asked)."""
    import contextlib

    @contextlib.contextmanager
    def limit():
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 1024) / total)
        held = []
        try:
            try:
                while True:  # what the allocator still holds in large blocks
                    held.append(torch.empty(2 << 20, dtype=torch.uint8, device=DEV))
            except torch.OutOfMemoryError:
                pass
            yield
        finally:
            held.clear()
            torch.cuda.set_per_process_memory_fraction(1.0)

    return limit


@pytest.mark.parametrize("path", ["compiled", "python"])
def test_out_of_memory_is_torch_out_of_memory(monkeypatch, no_memory, path):
    """A result that does not fit raises torch.OutOfMemoryError on both paths
    (what a serving loop catches to preempt a sequence), and the next call
    that fits works."""
    f16 = torch.float16
    z = torch.zeros(1, 1, 1, 64, dtype=f16, device=DEV)
    q = z.expand(64, 64, 128, 64)
    kp = torch.zeros(2048, 16, 64, 64, dtype=f16, device=DEV)
    bt, lens = torch.zeros(64, 16, dtype=torch.int32, device=DEV), torch.full((64,), 200, dtype=torch.int32, device=DEV)
    cache = PagedKVCache(KVCacheConfig(1, 8, 256, 1024, 16, f16, DEV))
    tables = [cache.new_sequence() for _ in range(64)]
    for t in tables:
        t.length = 100
    step = cache.prepare_step(tables, 32, num_heads=32)
    qs, ks = (torch.zeros(1, 1, 1, 256, dtype=f16, device=DEV).expand(64, h, 32, 256) for h in (32, 8))
    ks = ks.contiguous()
    one = cache.new_sequence()
    one.blocks, one.length = list(range(1000)), 16000
    x, w, s = (torch.zeros(16384, 16, dtype=f16, device=DEV), torch.zeros(2048, 16, dtype=torch.int8, device=DEV),
               torch.zeros(2048, dtype=f16, device=DEV))
    calls = {"flash": lambda: flash_attention(q, q, q), "paged": lambda: paged_attention(q, kp, kp, bt, lens),
             "prefill": lambda: paged_prefill(q, kp, kp, bt, lens),
             "section": lambda: attention_section(qs, ks, ks, 0, cache, step),
             "gather": lambda: cache.gather(0, one), "int8": lambda: int8_matmul(x, w, s)}
    with monkeypatch.context() as m:
        if path == "python":
            _python_only(m)
        for name, call in calls.items():
            with no_memory(), pytest.raises(torch.OutOfMemoryError):
                call()
            assert call() is not None, name


@pytest.mark.parametrize("path", ["compiled", "python"])
def test_split_launches_go_without_their_workspace(monkeypatch, no_memory, path):
    """Calls whose keys are split fit a full GPU: without room for the partial
    states they run unsplit."""
    g = torch.Generator().manual_seed(1)
    f16 = torch.float16
    q = torch.randn(1, 32, 300, 128, generator=g).to(DEV, f16)
    kp, vp = (torch.randn(400, 16, 8, 128, generator=g).to(DEV, f16) for _ in range(2))
    bt, lens = torch.arange(400, dtype=torch.int32, device=DEV).view(1, 400), torch.full((1,), 6400, dtype=torch.int32, device=DEV)
    k, v = (p.view(1, 6400, 8, 128).transpose(1, 2) for p in (kp, vp))
    out = torch.empty_like(q)
    assert _lib.load().cie_flash_workspace_bytes(1, 32, 8, 300, 6400, 128, 1, 0) > 4 << 20
    assert _lib.load().cie_flash_paged_workspace_bytes(1, 32, 8, 300, 128, 0, 16, 400, 0) > 4 << 20
    with monkeypatch.context() as m:
        if path == "python":
            _python_only(m)
        for call in (lambda: flash_attention(q, k, v, causal=True, out=out),
                     lambda: paged_prefill(q, kp, vp, bt, lens, out=out)):
            want = call().clone()
            with no_memory():
                got = call()
            assert (got.float() - want.float()).abs().max().item() <= 2e-3


def test_single_sequence_moves_are_not_captured():
    """append / gather of one sequence put host block ids into the launch: a
    graph would replay stale ones, so under capture the extension hands them
    back (the Python path's copy to the device then refuses)."""
    cache = PagedKVCache(KVCacheConfig(1, 2, 64, 8, 16, torch.float16, DEV))
    k = torch.ones(3, 2, 64, dtype=torch.float16, device=DEV)
    args = (k, k, cache.k[0], cache.v[0], [5], 0)
    x = torch.zeros(1, device=DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1)
        assert _lib.host().append_seq(*args) is None
        assert _lib.host().gather(cache.k[0], cache.v[0], [5], 3) is None
    graph.replay()
    torch.cuda.synchronize()
    assert x.item() == 1 and not cache.k[0].any()
    assert _lib.host().append_seq(*args) is True
    assert torch.equal(_lib.host().gather(cache.k[0], cache.v[0], [5], 3)[0], k)


def _workspace_calls(seed):
    """Calls that allocate a workspace each (key splits dense and paged, split
    K, paged partial states), as closures over inputs of their own, and the
    inputs to refill."""
    g = torch.Generator().manual_seed(seed)
    rand = lambda *shape: torch.randn(shape, generator=g).half().to(DEV)  # noqa: E731
    q, qp, qd = rand(1, 32, 5, 64), rand(1, 16, 300, 64), rand(3, 16, 1, 64)
    k, v = rand(1, 8, 3001, 64), rand(1, 8, 3001, 64)
    kp, vp = rand(300, 16, 4, 64), rand(300, 16, 4, 64)
    bt = torch.randperm(300, generator=g).int().to(DEV)
    lens = torch.tensor([1500, 700, 33], dtype=torch.int32, device=DEV)
    x, w = rand(96, 2048), torch.randint(-127, 128, (512, 2048), generator=g).to(torch.int8).to(DEV)
    sc = torch.rand(512, generator=g).half().to(DEV)
    lib = _lib.load()
    assert min(lib.cie_flash_workspace_bytes(1, 32, 8, 5, 3001, 64, 1, 0),
               lib.cie_flash_paged_workspace_bytes(1, 16, 4, 300, 64, 0, 16, 100, 0),
               lib.cie_int8_matmul_workspace_bytes(96, 512, 2048)) > 0
    calls = [lambda: flash_attention(q, k, v, causal=True),
             lambda: paged_prefill(qp, kp, vp, bt[:100].view(1, 100), lens[:1]),
             lambda: paged_attention(qd, kp, vp, bt.view(3, 100), lens),
             lambda: int8_matmul(x, w, sc, bias=sc)]
    return calls, (q, qp, qd, k, v, kp, vp, x)


def test_workspaces_in_a_captured_graph():
    """A graph of calls that allocate their workspaces, replayed with new
    inputs and eager calls in between."""
    calls, inputs = _workspace_calls(11)
    g = torch.Generator().manual_seed(12)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for call in calls:
            call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [call() for call in calls]
    for _ in range(3):
        for t in inputs:
            t.copy_(torch.randn(t.shape, generator=g).half())
        graph.replay()
        torch.cuda.synchronize()
        got = [o.clone() for o in outs]
        for a, call in zip(got, calls):
            assert torch.isfinite(a.float()).all() and torch.equal(a, call())


def test_two_threads_on_their_own_streams():
    """The extension releases the GIL around a launch: two threads, each on a
    stream of its own, get what one thread gets on the default stream."""
    import threading

    sets = [_workspace_calls(seed) for seed in (21, 22)]
    want = [[call() for call in calls] for calls, _ in sets]
    torch.cuda.synchronize()
    bad, gate = [], threading.Barrier(2)

    def work(i):
        try:
            stream = torch.cuda.Stream()
            gate.wait(timeout=30)
            with torch.cuda.stream(stream):
                for _ in range(25):
                    got = [call() for call in sets[i][0]]
                    stream.synchronize()
                    bad.extend((i, n) for n, (a, b) in enumerate(zip(got, want[i])) if not torch.equal(a, b))
        except Exception as e:  # noqa: BLE001
            bad.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not any(t.is_alive() for t in threads) and not bad, bad[:4]
