"""Side-stream execution of the per-layer dot-product kernels, overlapped with the rest of
the backward pass.

The backward hook of a layer with enough work to overlap enqueues its kernels on a second
HIP stream (default priority) after that stream has waited for everything the autograd
stream enqueued so far.  The hook's input tensors are marked as in use by the side stream, so
the caching allocator does not hand their memory back to the autograd stream before the side
kernels finish.
At the end of the backward pass an autograd-engine callback makes the autograd stream wait
for the side stream, so the optimizer, the engines' aggregation and any host copy see
finished results.  ``join(device)`` does the same wait explicitly (the engines call it
before reading results, which also covers a backward pass that raised).

Memory written on the side stream and later read on the autograd stream needs no extra
bookkeeping: every later side-stream launch is preceded by a wait on the autograd stream.
A train gradient that one layer stored on the autograd stream and another adds to on the side
stream (or the other way round) is kept by its parameter until after that wait, and the adding
layer joins first.
"""
from __future__ import annotations

import threading
from typing import Dict

import torch

_lock = threading.Lock()
_streams: Dict[int, torch.cuda.Stream] = {}
_join_queued: Dict[int, bool] = {}
_events = threading.local()   # per thread: {device index: the event of _wait}

enabled = True


def side_stream(device: torch.device) -> torch.cuda.Stream:
    idx = device.index if device.index is not None else torch.cuda.current_device()
    with _lock:
        s = _streams.get(idx)
        if s is None:
            s = torch.cuda.Stream(device=idx)   # default priority
            _streams[idx] = s
    return s


def _wait(idx: int, waiter: torch.cuda.Stream, on: torch.cuda.Stream) -> None:
    """`waiter` waits for what `on` holds so far, through one event kept per thread and device (a
    wait refers to the record before it; recording again does not reach earlier waits).  Under
    graph capture the event belongs to the graph, so each wait takes its own."""
    if torch.cuda.is_current_stream_capturing():
        waiter.wait_stream(on)
        return
    events = _events.__dict__.setdefault("by_device", {})
    ev = events.get(idx)
    if ev is None:
        ev = events[idx] = torch.cuda.Event()
    ev.record(on)
    ev.wait(waiter)


def join(device=None) -> None:
    """The current stream of `device` waits for the side stream's work so far."""
    if not _streams:
        return
    devices = [device] if device is not None else [torch.device("cuda", i) for i in _streams]
    for dev in devices:
        dev = torch.device(dev)
        if dev.type != "cuda":
            continue
        idx = dev.index if dev.index is not None else torch.cuda.current_device()
        s = _streams.get(idx)
        if s is not None:
            torch.cuda.current_stream(idx).wait_stream(s)
        _join_queued.pop(idx, None)


def _queue_join(idx: int, cur: torch.cuda.Stream, side: torch.cuda.Stream) -> None:
    if _join_queued.get(idx):
        return

    def _end_of_backward():
        cur.wait_stream(side)
        _join_queued.pop(idx, None)

    try:
        torch.autograd.Variable._execution_engine.queue_callback(_end_of_backward)
        _join_queued[idx] = True
    except RuntimeError:
        # Not inside a backward pass: order the side work before anything enqueued later.
        cur.wait_stream(side)
        _join_queued.pop(idx, None)


class on_side_stream:
    """``with on_side_stream(*tensors):`` runs the body on the side stream of the tensors' device
    (no-op on CPU or when disabled).  The tensors are the body's inputs produced on the current
    stream."""

    __slots__ = ("_tensors", "_idx", "_cur", "_side", "_ctx")

    def __init__(self, *tensors):
        self._tensors = tensors
        self._side = self._ctx = None

    def __enter__(self):
        ts = [t for t in self._tensors if isinstance(t, torch.Tensor)]
        if not enabled or not ts or ts[0].device.type != "cuda":
            return self
        dev = ts[0].device
        here = torch.cuda.current_device()
        self._idx = idx = dev.index if dev.index is not None else here
        side = side_stream(dev)
        self._cur = torch.cuda.current_stream(idx)
        _wait(idx, side, self._cur)
        for t in ts:
            t.record_stream(side)
        if here == idx:
            # Same device: switch the current stream only (the stream context manager also
            # saves and restores the current device, several times the cost per hook).
            torch.cuda.set_stream(side)
        else:
            self._ctx = torch.cuda.stream(side)
            self._ctx.__enter__()
        self._side = side
        return self

    def __exit__(self, exc_type, exc, tb):
        if self._side is None:
            return False
        if self._ctx is not None:
            self._ctx.__exit__(exc_type, exc, tb)
        else:
            torch.cuda.set_stream(self._cur)
        if exc_type is None:
            _queue_join(self._idx, self._cur, self._side)
        return False
