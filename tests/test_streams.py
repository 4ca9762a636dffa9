"""Kept device data across streams, with streams and events stood in for on
the CPU: who waits for what, and which buffers a training step writes."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from multics_amd import _capi, _ready, hier_masks, rope
from multics_amd import metadata as M


@pytest.fixture
def gpu(monkeypatch):
    """CPU tensors taken for a GPU's: ``gpu.stream`` is the current stream,
    ``gpu.log`` gets ("record", stream) and ("wait", stream, recorded on)."""
    state = SimpleNamespace(stream=1, log=[], capturing=False, used=[])

    class Stream:
        def __init__(self):
            self.cuda_stream = state.stream

        def wait_event(self, e):
            state.log.append(("wait", state.stream, e.on))

    class Event:
        on = None

        def record(self, s):
            self.on = s.cuda_stream
            state.log.append(("record", s.cuda_stream))

    def tensors(x):
        if torch.is_tensor(x):
            yield SimpleNamespace(device=SimpleNamespace(type="cuda"), record_stream=lambda s: state.used.append(
                (x.data_ptr(), s.cuda_stream)))
        elif isinstance(x, (tuple, list)):
            for v in x:
                yield from tensors(v)
        elif isinstance(x, dict):
            yield from tensors(list(x.values()))
        elif hasattr(x, "kept_tensors"):
            yield from tensors(x.kept_tensors())

    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: Stream())
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(_capi, "stream_of", lambda d: state.stream)
    monkeypatch.setattr(_ready, "device_tensors", tensors)
    monkeypatch.setattr(_ready, "capturing", lambda d: state.capturing)
    for mod, name in ((M, "_META_CACHE"), (M, "_LAYOUT_CACHE"), (M, "_PLAN_LRU"),
                      (hier_masks, "_MASK_CACHE"), (rope, "_COS_SIN_CACHE")):
        monkeypatch.setattr(mod, name, type(getattr(mod, name))())
    return state


def _list(n=1):
    z = lambda *s: torch.zeros(*s, dtype=torch.int32)
    return M.TileList(items=z(n, 8), kv_idx=z(64), kv_mask=z(64), blk_and=z(1), n_items=n,
                      item_ranges=(), logical_pairs=0)


def test_a_kept_entry_is_waited_for_once_per_stream(gpu):
    cache = type(M._META_CACHE)()
    t = _list()
    M._lru_put(cache, "k", t, "WAN_HIER_SEGMENTED_META_CACHE_SIZE", "64")
    assert gpu.log == [("record", 1)]
    assert M._lru_get(cache, "k") is t and len(gpu.log) == 1      # its own stream: nothing
    gpu.stream = 2
    for _ in range(3):
        assert M._lru_get(cache, "k") is t
    assert gpu.log[1:] == [("wait", 2, 1)]
    assert {p for p, s in gpu.used if s == 2} >= {t.items.data_ptr(), t.kv_idx.data_ptr(),
                                                  t.kv_mask.data_ptr(), t.blk_and.data_ptr()}
    gpu.stream = 1
    M._lru_get(cache, "k")
    assert len(gpu.log) == 2


def test_capture_waits_for_nothing_and_keeps_nothing(gpu):
    cache = type(M._META_CACHE)()
    t = _list()
    M._lru_put(cache, "k", t, "WAN_HIER_SEGMENTED_META_CACHE_SIZE", "64")
    gpu.stream, gpu.capturing = 2, True
    assert M._lru_get(cache, "k") is t and gpu.log == [("record", 1)]
    M._lru_put(cache, "made in a graph", _list(), "WAN_HIER_SEGMENTED_META_CACHE_SIZE", "64")
    assert list(cache) == ["k"]
    rope.freqs_to_cos_sin(torch.ones(3, 1, 2, dtype=torch.complex64))
    assert not rope._COS_SIN_CACHE
    gpu.capturing = False                              # an eager call on it does wait
    M._lru_get(cache, "k")
    assert gpu.log[-1] == ("wait", 2, 1)


def test_lists_derived_from_a_kept_list(gpu, monkeypatch):
    """Key-major and launch lists are made on the stream that first asks;
    a list that nobody keeps (a training step's) records nothing."""
    t = _list()
    t.__dict__["_ready"] = _ready.made(t)
    gpu.stream = 2
    monkeypatch.setattr(M, "transpose_tiles_host", lambda tiles: _list())
    kt, _ = M.backward_lists(t)
    M._derived_on(t, kt)                               # (the device path's line)
    run = M._set_launch(t, _list().items, None)
    gpu.log.clear()
    assert M.backward_lists(t)[0] is kt and M.transpose_tiles(t) is kt and M.launch_list(t) is run
    assert gpu.log == []
    gpu.stream = 3
    assert M.transpose_tiles(t) is kt and M.backward_lists(t)[0] is kt
    assert M.launch_list(t) is run
    assert gpu.log == [("wait", 3, 2), ("wait", 3, 2)]
    gpu.log.clear()
    step = _list()
    M._set_launch(step, _list().items, None)
    gpu.stream = 4
    M.launch_list(step)
    assert gpu.log == []


def test_tables_and_masks(gpu):
    # (cos / sin tables are a stream's own)
    f = SimpleNamespace(device=torch.device("cuda", 0), _version=0, requires_grad=False,
                        shape=(3, 1, 2), reshape=lambda *a: torch.ones(3, 2, dtype=torch.complex64))
    a = rope.freqs_to_cos_sin(f)
    assert rope.freqs_to_cos_sin(f)[0] is a[0]
    gpu.stream = 2
    assert rope.freqs_to_cos_sin(f)[0] is not a[0] and gpu.log == []
    hier_masks._cache_put("k", (_list(), 1, 1))
    gpu.stream = 3
    M._lru_get(hier_masks._MASK_CACHE, "k")
    assert gpu.log == [("record", 2), ("wait", 3, 2)]


def _plan(monkeypatch, calls):
    sup = _list(2)
    sup._layout = (np.zeros(4, np.int64), np.zeros(4, np.int64))
    sup.row_extent = sup.key_extent = 128
    sup.n_groups = sup.frames_per_group = 1
    monkeypatch.setattr(M, "build", lambda *a, **k: SimpleNamespace(tiles=sup))
    monkeypatch.setattr(M, "backward_lists", lambda *a: (_list(), None))

    def call(name, *args):
        a = args[0]._obj
        calls.append((name, args[-1], {f: getattr(a, f) for f, _ in a._fields_
                                       if f in ("membership", "global_only", "q_active",
                                                "local_active", "ws", "totals")}))

    monkeypatch.setattr(_capi, "call", call)
    return M.MembershipLogitsPlan(device="cpu", P=2, T=2, L=4, N=1, KL=1, KG=1, n=1, window=1,
                                  direct=True)


def test_steps_on_two_streams_write_their_own_buffers(gpu, monkeypatch):
    calls = []
    plan = _plan(monkeypatch, calls)
    logits = torch.ones(2, 1, 2)

    def step(stream):
        gpu.stream = stream
        calls.clear()
        t = plan.build(logits)
        written = {}
        for name, on, ptrs in calls:
            assert on == stream or getattr(on, "value", on) == stream, name
            written.update(ptrs)
        return t, written

    keep = [step(1), step(2), step(1), step(2)]
    a, b, a2, b2 = (w for _, w in keep)
    assert set(a) == {"membership", "global_only", "q_active", "local_active", "ws", "totals"}
    assert a == a2 and b == b2                       # a stream's buffers are kept
    assert all(a[f] != b[f] for f in a)              # and are its own
    assert gpu.log.count(("wait", 2, 1)) == 1        # the plan itself, once
    keep += [step(s) for s in range(3, 30)]
    assert len(plan._steps) == M._PLAN_STREAMS
    gpu.capturing = True                             # a graph's buffers are nobody else's
    t, g = step(1)
    assert all(g[f] != a[f] for f in a) and t._keepalive[1].ws.data_ptr() == g["ws"]


def test_threads_share_a_small_cache(monkeypatch):
    """Lookups move entries that other threads evict meanwhile."""
    import sys
    import threading
    monkeypatch.setenv("WAN_HIER_SEGMENTED_META_CACHE_SIZE", "1")
    cache, errors = type(M._META_CACHE)(), []

    def work(i):
        try:
            for j in range(20000):
                k = (i + j) % 3
                v = M._lru_get(cache, k)
                assert v is None or v == ("value", k)
                M._lru_put(cache, k, ("value", k), "WAN_HIER_SEGMENTED_META_CACHE_SIZE", "64")
        except BaseException as e:      # noqa: B036 (reported below)
            errors.append(e)

    old = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(old)
    assert not errors and len(cache) <= 1
