"""Kept lists and plans used from several streams on the GPU.  The lists are
compared on the host, never launched on."""

import numpy as np
import pytest
import torch

from multics_amd import _capi
from multics_amd import metadata as M
from tests.gpu_util import need_gpu, say

pytestmark = pytest.mark.gpu
GEO = dict(P=3, T=6, L=20, N=2, KL=2, KG=3, n=2, window=4, direct=True)
SLEEP = 20_000_000      # cycles: well above the time of a build


def _arrays(t):
    """What a launch reads: the items, the cut items and the lists that the
    items address (entries between the lists are not written)."""
    n = t.n_items
    items, cut, idx, msk, blk = (x.cpu() for x in (t.items[:n], M.launch_list(t).items[:n],
                                                   t.kv_idx, t.kv_mask, t.blk_and))
    return [items, cut] + [x for o, c in items[:, 5:7].tolist()
                           for x in (idx[o:o + c], msk[o:o + c], blk[o // 64:(o + c) // 64])]


def _same(got, want):
    assert len(got) == len(want)
    for i, (x, y) in enumerate(zip(got, want)):
        assert torch.equal(x, y), i


def _tiles():
    labels = np.array([[0, 1, 0]] * GEO["T"])
    return M.full_sequence_tiles(device="cuda", labels=labels,
                                 active=np.ones((GEO["T"], GEO["N"]), bool), **GEO)


def test_a_list_found_from_another_stream_is_complete(monkeypatch):
    """The last launches of a build wait behind a long kernel on the first
    stream; a second stream finds the list meanwhile and reads it."""
    need_gpu()
    say("list found from another stream")
    M._LAYOUT_CACHE.clear()
    want = _arrays(_tiles())
    M._LAYOUT_CACHE.clear()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    call = _capi.call

    def slow(name, *args):
        if name in ("hier_meta_build", "hier_derive_build"):
            torch.cuda._sleep(SLEEP)
        call(name, *args)

    monkeypatch.setattr(_capi, "call", slow)
    with torch.cuda.stream(a):
        t = _tiles()
    monkeypatch.setattr(_capi, "call", call)
    with torch.cuda.stream(b):
        hit = _tiles()
        assert hit is t
        got = _arrays(hit)                  # copies on b, waiting for b alone
    _same(got, want)
    # the key-major list, made by a's first backward, found by b's
    monkeypatch.setattr(_capi, "call", slow)
    with torch.cuda.stream(a):
        kt = M.backward_lists(t)[0]
    monkeypatch.setattr(_capi, "call", call)
    with torch.cuda.stream(b):
        assert M.backward_lists(t)[0] is kt
        got = _arrays(kt)
    torch.cuda.synchronize()
    _same(got, _arrays(kt))
    assert int(kt.items[:, 6].sum()) > 0


def test_a_list_dropped_while_another_stream_reads_it():
    """Its memory is not handed out before that stream has read it."""
    need_gpu()
    say("list dropped while read")
    M._LAYOUT_CACHE.clear()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        t = _tiles()
    torch.cuda.synchronize()
    want = _arrays(t)[2]
    with torch.cuda.stream(b):
        hit = _tiles()
        torch.cuda._sleep(SLEEP)
        copy = hit.kv_idx.clone()
    shape, (off, cnt) = t.kv_idx.shape, t.items[0, 5:7].tolist()
    M._LAYOUT_CACHE.clear()
    del t, hit
    with torch.cuda.stream(a):
        later = [torch.full(shape, -1, dtype=torch.int32, device="cuda") for _ in range(64)]
    torch.cuda.synchronize()
    assert torch.equal(copy.cpu()[off:off + cnt], want) and len(later) == 64


def test_steps_of_one_plan_on_two_streams():
    """Lists built from logits on two streams in turn, with nothing between
    them, are those of a build by itself."""
    need_gpu()
    say("steps on two streams")
    g = torch.Generator().manual_seed(2)
    plan = M.MembershipLogitsPlan(device="cuda", **GEO)
    logits = [torch.randn(GEO["T"], GEO["N"], GEO["P"], generator=g).cuda() for _ in range(12)]
    want = []
    for lg in logits:
        t = plan.build(lg)
        torch.cuda.synchronize()
        want.append(t)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for s in streams:
        with torch.cuda.stream(s):
            torch.cuda._sleep(SLEEP)        # so that the steps pile up and run side by side
    for i, lg in enumerate(logits):
        with torch.cuda.stream(streams[i % 2]):
            got.append(plan.build(lg))
    torch.cuda.synchronize()

    for t, w in zip(got, want):
        _same(_arrays(t), _arrays(w))
        _same(_arrays(M.transpose_tiles(t)), _arrays(M.transpose_tiles(w)))


def test_a_step_captured_in_a_graph_replays():
    """A step's lists made in a graph follow the logits on every replay, with
    eager steps of the same plan between."""
    need_gpu()
    say("captured step")
    g = torch.Generator().manual_seed(3)
    plan = M.MembershipLogitsPlan(device="cuda", **GEO)
    logits = torch.randn(GEO["T"], GEO["N"], GEO["P"], generator=g).cuda()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        plan.build(logits)                  # warm-up, as graph users do
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        t = plan.build(logits)
    for i in range(4):
        logits.copy_(torch.randn(logits.shape, generator=g))
        graph.replay()
        plan.build(-logits)                 # another membership, eagerly
        torch.cuda.synchronize()
        w = plan.build(logits)
        torch.cuda.synchronize()
        _same(_arrays(t), _arrays(w))
        _same(_arrays(M.transpose_tiles(t)), _arrays(M.transpose_tiles(w)))
