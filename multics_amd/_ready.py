"""Device data that is kept and handed out again -- work lists, plans, tables --
across streams and threads.

A kept entry is made by launches on the stream of the call that missed it; a
later call may find it from another stream, before those launches have run,
and its memory may go back to the first stream's pool while the second still
reads it.  ``Ready`` is the event behind the launches that made an entry:
``join`` makes the current stream wait for it and tells the allocator that the
stream uses the memory, once per stream, and is a set lookup after that (and
always on the stream that made it).

Under graph capture an entry is used as it is (a wait for work outside a
capture is an error; ``torch.cuda.graph`` synchronizes the device before it
captures) and nothing made is kept: it holds nothing until the graph runs."""

from __future__ import annotations

import dataclasses

import torch

from . import _capi


def touch(cache, key) -> None:
    """Moves a kept entry to the end of its ordered dictionary, unless another
    thread has evicted it since it was found."""
    try:
        cache.move_to_end(key)
    except KeyError:
        pass


def evict(cache, n: int) -> None:
    """Drops the oldest entries until at most ``n`` are left (several threads
    may, and then drop no more than one too many each)."""
    while len(cache) > n:
        try:
            cache.popitem(last=False)
        except KeyError:
            return


def capturing(device) -> bool:
    return device is not None and device.type == "cuda" and torch.cuda.is_current_stream_capturing()


def device_tensors(x):
    """The GPU tensors of a kept value: a tensor, a dataclass, an object with
    ``kept_tensors()``, or tuples, lists and dicts of them."""
    if torch.is_tensor(x):
        if x.is_cuda:
            yield x
    elif isinstance(x, (tuple, list)):
        for v in x:
            yield from device_tensors(v)
    elif isinstance(x, dict):
        yield from device_tensors(list(x.values()))
    elif hasattr(x, "kept_tensors"):
        yield from device_tensors(x.kept_tensors())
    elif dataclasses.is_dataclass(x):
        for f in dataclasses.fields(x):
            yield from device_tensors(getattr(x, f.name))


class Ready:
    __slots__ = ("device", "event", "streams")

    def __init__(self, device):
        stream = torch.cuda.current_stream(device)
        self.device = device
        self.event = torch.cuda.Event()
        self.event.record(stream)
        self.streams = {stream.cuda_stream}

    def join(self, value) -> None:
        """The current stream may use ``value``, made where this was recorded."""
        handle = _capi.stream_of(self.device)
        if handle in self.streams or capturing(self.device):
            return
        stream = torch.cuda.current_stream(self.device)
        stream.wait_event(self.event)
        for t in device_tensors(value):
            t.record_stream(stream)
        self.streams.add(handle)


def being_captured(value) -> bool:
    """Whether the value's launches go into a graph (it is not to be kept)."""
    t = next(device_tensors(value), None)
    return t is not None and capturing(t.device)


def made(value):
    """``Ready`` of a value that launches on the current stream have just
    made; None if it holds no GPU tensor."""
    t = next(device_tensors(value), None)
    return None if t is None else Ready(t.device)
