"""Two-launch plans of long transforms (fft/long.py): the cut, the tiles' addresses and the
twiddle tables, restated in NumPy on the CPU."""
import numpy as np
import pytest

from vkdispatch_amd.fft import long as LG
from vkdispatch_amd.fft.planner import LDS_BYTES_MAX, slots

LENGTHS = [1 << 15, 1 << 20, 1 << 21, 59049, 25200, 120120, 463050, 864360, 823543, 16807 * 2, 11 ** 3 * 13]


def _outer_roots(rows, cols, step, n):
    """vkx_outer_roots in NumPy."""
    r, c = np.arange(rows)[:, None], np.arange(cols)[None, :]
    return np.exp(-2j * np.pi * (r * c * step % n) / n)


@pytest.mark.parametrize("n", LENGTHS)
def test_tiles_stay_in_bounds(n):
    n1, n2 = LG.split_length(n)
    assert n1 * n2 == n
    for m, across, turned in ((n1, n2, True), (n2, n1, False)):
        for batch in (1, 300):
            t = LG.tile_plan(m, across, batch, turned)
            assert np.prod(t.radices) == m and len(t.radices) >= 2
            assert t.lds_bytes <= LDS_BYTES_MAX and t.TT * t.B <= 1024
            assert max(slots(m, r, t.TT) for r in t.radices) <= LG.MAX_RADIX
            # LDS positions (b, pos): all different, all inside (vkx_long.h tile_addr)
            pos, b = np.arange(m)[:, None], np.arange(t.B)[None, :]
            addr = pos * t.pitch + b + pos // t.radices[0] * t.B
            assert len(np.unique(addr)) == m * t.B and addr.max() < t.lds_elems


@pytest.mark.parametrize("n", [n for n in LENGTHS if n <= 1 << 17])
def test_two_launches_are_the_transform(n):
    n1, n2 = LG.split_length(n)
    rows = LG.tile_plan(n2, n1, 1, False)
    radix = LG.tile_plan(n1, n2, 1, True).radices[-1]
    w = n1 // radix
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    cols = np.fft.fft(x.reshape(n1, n2), axis=0)
    k1 = np.arange(n1)
    a, rot = _outer_roots(n2, w, 1, n), _outer_roots(n2, radix, w, n)
    tw = a[:, k1 % w] * rot[:, k1 // w]               # [j2][k1], as the column kernel multiplies
    y = np.full(LG.scratch_points(n, rows.B), np.nan, complex)
    j2 = np.arange(n2)[:, None]
    at = ((k1 // rows.B) * n2 + j2) * rows.B + k1 % rows.B
    assert at.max() < y.size and len(np.unique(at)) == n
    y[at] = cols.T * tw
    out = np.empty(n, complex)
    for tile in range(-(-n1 // rows.B)):
        block = y[tile * n2 * rows.B:(tile + 1) * n2 * rows.B].reshape(n2, rows.B)
        for b in range(min(rows.B, n1 - tile * rows.B)):
            out[np.arange(n2) * n1 + tile * rows.B + b] = np.fft.fft(block[:, b])
    ref = np.fft.fft(x)
    assert np.linalg.norm(out - ref) <= 1e-12 * np.linalg.norm(ref)


def test_what_does_not_split():
    """Prime factors above 13, short lengths and lengths beyond two tiles stay elsewhere."""
    for n in (17 * 1024, 65537, 2048, 1 << 26):
        assert LG.split_length(n) is None


def test_scratch_of_streams_and_captures(monkeypatch):
    """Two streams never share what lies between the launches, nor do a capture and the
    launches that follow it; what a plan keeps is bounded."""
    import threading
    capturing = set()
    monkeypatch.setattr(LG, "Buffer", lambda shape, dtype: object())
    monkeypatch.setattr(LG.rt, "is_capturing", lambda s=None: s in capturing)
    plan = object.__new__(LG.LongFFT)
    plan._points, plan._scratch, plan._captured, plan._lock = 8, {}, None, threading.Lock()
    got = {s: plan._scratch_for(s) for s in range(7)}
    assert len({id(b) for b in got.values()}) == 7 and len(plan._scratch) == LG.SCRATCH_STREAMS
    assert plan._scratch_for(6) is got[6] and plan._scratch_for(0) is not got[0]
    for stream in (6, 99):  # warmed up on this stream, and not
        plan._captured = None
        capturing = {stream}
        taken = plan._scratch_for(stream)
        assert plan._scratch_for(stream) is taken
        capturing = set()
        assert all(plan._scratch_for(s) is not taken for s in range(7)) and plan._scratch_for(stream) is not taken
