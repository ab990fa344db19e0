"""What the launches of one call hand to each other in device memory.

It belongs to one sequence of launches at a time, so work that can overlap never shares it:

* a call takes the buffer of its stream, which all plans share (work on a stream runs in
  order) and which grows to the largest of them; it holds ``launch_order`` while it
  enqueues, so that another thread's launches on that stream do not come in between;
* a CommandGraph takes that of the stream it is submitted on, when it is captured for it
  (the graph then runs on this stream only);
* inside a capture of the caller's, whose replays may run at any time and on any stream, a call
  takes a buffer that its plan keeps for this capture, and a CommandGraph one that it keeps;
* a launch that is bound to be run later, on any stream, has a buffer of its own.

A buffer that is let go is freed by hipFree, which waits for the work in flight.
"""
from __future__ import annotations

import threading
from typing import Dict, List, Tuple

from .. import runtime as rt
from ..buffer import Buffer
from .shader_factories import register_plan_cache

SCRATCH_STREAMS = 6    # streams whose buffers are kept; while calls alternate between more, each frees the
#                        oldest (a wait for the GPU) and allocates
SCRATCH_CAPTURES = 16  # captures of a plan with a buffer of their own; the next one takes the oldest's, and
#                        replays of those two must not overlap

_streams: Dict[object, Tuple[int, object]] = {}
_streams_lock = threading.Lock()
_pinned: List[object] = []
_order = threading.RLock()


def launch_order():
    """Held while a call enqueues launches that use its stream's scratch: another thread's on
    this stream must not come in between."""
    return _order


def pin(owner) -> None:
    """Keep what a capture of the caller's launches with, whatever drops it, until clear()."""
    if not any(o is owner for o in _pinned):
        _pinned.append(owner)


class StreamScratch:
    """Owner of launches with ``_points`` complex64 values between them."""

    def _init_scratch(self, points: int) -> None:
        self._points = int(points)
        self._scratch, self._lock = _streams, _streams_lock
        self._captured: Dict[tuple, object] = {}

    def _new_scratch(self) -> Buffer:
        with rt.allocating_in_capture():
            return Buffer((self._points,))

    def _scratch_for(self, stream: int):
        """The buffer of a call on ``stream``, to be used under ``launch_order()``."""
        with self._lock:
            if rt.is_capturing(stream):
                return self._scratch_of_capture(stream)
            kept, key = self._scratch, rt.stream_key(stream)
            have = kept.get(key)
            if have is None or have[0] < self._points or next(reversed(kept)) != key:
                kept.pop(key, None)
                if have is None or have[0] < self._points:
                    have = (self._points, self._new_scratch())
                kept[key] = have  # the newest comes last
                while len(kept) > SCRATCH_STREAMS:
                    del kept[next(iter(kept))]
            return have[1]

    def _scratch_of_capture(self, stream: int):
        kept = self._captured = self._captured or {}
        # the branches of one capture may overlap, too
        key = (rt.capture_id(stream), rt.stream_key(stream), self._points)
        if key not in kept:
            full = len(kept) >= SCRATCH_CAPTURES
            oldest = next((k for k in kept if k[2] >= self._points), None) if full else None
            kept[key] = self._new_scratch() if oldest is None else kept.pop(oldest)
            pin(self)
        return kept[key]


def clear() -> None:
    """Let go of the buffers of calls and captures (graphs and bound launches hold theirs)."""
    with _streams_lock:
        _streams.clear()
        _pinned.clear()


register_plan_cache(clear)
