"""What the launches of one call hand to each other in device memory.

It belongs to one sequence of launches at a time, so work that can overlap never shares it:

* a call takes the buffer of its stream, which all plans share (work on a stream runs in
  order) and which grows to the largest of them; it holds ``launch_order`` while it
  enqueues, so that another thread's launches on that stream do not come in between;
* launches that are kept and run later, on any stream, have a buffer of their own, or that of
  the CommandGraph that they are recorded into (``CommandGraph.scratch``);
* a call inside a capture of the caller's takes a buffer that its plan keeps for this
  capture: the replays may run at any time and on any stream.

A buffer that is let go is freed by hipFree, which waits for the work in flight.
"""
from __future__ import annotations

import threading
from typing import Dict, List, Tuple

from .. import runtime as rt
from .shader_factories import register_plan_cache

SCRATCH_STREAMS = 6    # streams whose buffers are kept; while calls alternate between more, each frees the
#                        oldest (a wait for the GPU) and allocates
SCRATCH_CAPTURES = 16  # captures of a plan with a buffer of their own; the next one takes the oldest's, and
#                        replays of those two must not overlap

_streams: Dict[object, Tuple[int, object]] = {}
_streams_lock = threading.Lock()
_pinned: List[object] = []
_order = [threading.RLock() for _ in range(16)]
_PER_THREAD_STREAM = 2  # hipStreamPerThread: one handle for a stream of each thread


def _stream_key(stream: int):
    return (stream, threading.get_ident()) if stream == _PER_THREAD_STREAM else stream


def launch_order(stream: int):
    """Held while a call enqueues its launches on ``stream``: they use the stream's scratch,
    and another thread's must not come in between."""
    return _order[hash(_stream_key(stream)) % len(_order)]


class StreamScratch:
    """A plan with ``_points`` complex64 values between its launches; ``_new_scratch()`` allocates
    them."""

    def _init_scratch(self) -> None:
        self._scratch, self._lock = _streams, _streams_lock
        self._captured: Dict[tuple, object] = {}

    def _scratch_for(self, stream: int):
        """The buffer of a call on ``stream``, to be used under ``launch_order(stream)``."""
        with self._lock:
            if rt.is_capturing(stream):
                return self._scratch_of_capture(stream)
            key = _stream_key(stream)
            have = self._scratch.pop(key, None)
            if have is None or have[0] < self._points:
                have = (self._points, self._new_scratch())
            self._scratch[key] = have  # the newest comes last
            while len(self._scratch) > SCRATCH_STREAMS:
                del self._scratch[next(iter(self._scratch))]
            return have[1]

    def _scratch_of_capture(self, stream: int):
        kept = self._captured = self._captured or {}
        key = (rt.capture_id(stream), _stream_key(stream))  # the branches of one capture may overlap, too
        if key not in kept:
            kept[key] = self._new_scratch() if len(kept) < SCRATCH_CAPTURES else kept.pop(next(iter(kept)))
            if self not in _pinned:
                _pinned.append(self)  # a plan cache may drop the plan; the captured graph needs its memory
        return kept[key]


def clear() -> None:
    """Let go of the buffers of calls and captures (graphs and bound launches keep theirs)."""
    with _streams_lock:
        _streams.clear()
        _pinned.clear()


register_plan_cache(clear)
