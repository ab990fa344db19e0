"""Who shares what lies between the launches of one call: kernels and buffers that only note
what is done with them, on the CPU."""
import threading

import pytest

from vkdispatch_amd import dtypes as dt
from vkdispatch_amd import graph as G
from vkdispatch_amd import runtime as rt
from vkdispatch_amd.fft import functions as F
from vkdispatch_amd.fft import fused as FU
from vkdispatch_amd.fft import long as LG
from vkdispatch_amd.fft import mixed as MX
from vkdispatch_amd.fft import scratch


class _Kernel:
    def __init__(self, log, name):
        self.log, self.name = log, name

    def handle(self):
        return 1

    def bind(self, values):
        return [v.ptr for v in values], b""

    def launch(self, values, stream):
        self.launch_raw(*self.bind(values), stream)

    def launch_raw(self, ptrs, consts=b"", stream=None):
        self.log.append((self.name, rt.current_stream() if stream is None else stream, tuple(ptrs)))


class _Data:
    def __init__(self, ptr, size=1 << 20):
        self.ptr, self.size = ptr, size


@pytest.fixture
def device(monkeypatch):
    """The allocator's addresses, the current stream and what is being captured, as the
    test sets them; freed addresses are listed."""
    class Device:
        stream, capturing, freed, next_ptr = 1, {}, [], 1 << 20
    dev = Device()
    dev.capturing, dev.freed = {}, []

    def malloc(nbytes):
        dev.next_ptr += 1 << 20
        return dev.next_ptr
    monkeypatch.setattr(rt, "malloc", malloc)
    monkeypatch.setattr(rt, "free", dev.freed.append)
    monkeypatch.setattr(rt, "synchronize", lambda stream=None: None)
    monkeypatch.setattr(rt, "current_stream", lambda: dev.stream)
    monkeypatch.setattr(rt, "is_capturing", lambda s=None: (dev.stream if s is None else s) in dev.capturing)
    monkeypatch.setattr(rt, "lib", lambda: dev)
    dev.vkx_graph_begin = lambda s: dev.capturing.update({s: 1000 + s}) or 0
    dev.vkx_graph_end = lambda s, h: dev.capturing.pop(s) and 0
    dev.vkx_graph_launch = dev.vkx_graph_destroy = lambda *a: 0
    monkeypatch.setattr(rt, "capture_id", lambda s: dev.capturing.get(s, 0), raising=False)
    return dev


def _long_plan(points=64):
    """A LongFFT of 3 transforms in two chunks, its kernels noting their launches."""
    log = []
    plan = object.__new__(LG.LongFFT)
    cols, rows = _Kernel(log, "cols"), _Kernel(log, "rows")
    plan.n, plan.count, plan.chunks = 16, 3, [(0, 2), (2, 1)]
    plan.kernels = {1: (cols, rows), 2: (cols, rows)}
    plan.tables = (_Data(5), _Data(6))
    plan._points, plan._scratch, plan._captured, plan._lock = points, {}, None, threading.Lock()
    return plan, log


def _between(log):
    """(stream, scratch address) of every pair of launches, which must be the same in both."""
    out = []
    for (a, s, p), (b, t, q) in zip(log[::2], log[1::2]):
        assert (a, b) == ("cols", "rows") and s == t and p[0] == q[1]
        out.append((s, p[0]))
    return out


def _long(monkeypatch):
    """fft() of a long length as functions.py routes it."""
    plan, log = _long_plan()
    plan._init_scratch(64)
    monkeypatch.setattr(F, "_uniform_plan", lambda *a: plan)

    def call(buf, graph):
        assert F._large_or_prime_fallback((buf,), (3, 1 << 20), None, False, True, False, None, None, dt.complex64,
                                          dt.complex64, None, graph)
    return plan, log, call, _between


def _conv(monkeypatch):
    """convolve2DR of square images."""
    log = []
    plan = FU.Conv2DPhases(3, 256, 256)
    plan.kernels_ = [_Kernel(log, n) for n in ("rows", "cols", "irows")]
    plan._checked = True
    monkeypatch.setattr(FU, "fused_eligible", lambda *a, **kw: plan)

    def call(buf, graph):
        assert FU.try_convolve2DR(buf, _Data(77), graph)

    def between(log):
        out = []
        for three in zip(log[::3], log[1::3], log[2::3]):
            assert [n for n, _, _ in three] == ["rows", "cols", "irows"]
            (key,) = {(s, p[2]) for _, s, p in three}
            assert all(p[1] == 77 and p[5] == p[2] + 8 * 2 * 256 * 256 for _, _, p in three)  # two pairs, then Kt
            out.append(key)
        return out
    return plan, log, call, between


def _mixed(monkeypatch, passes=2):
    """fft3_mixed, two passes with one volume between them or three with two."""
    log = []
    plan = MX.Mixed3D((256, 256, 256), dt.complex_bf16, passes=passes)
    plan.passes = [_Kernel(log, str(n)) for n in range(passes)]
    monkeypatch.setattr(MX, "_plan", lambda *a: plan)

    def call(buf, graph):
        out = _Data(buf.ptr + 8)
        buf.shape = out.shape = (256, 256, 256)
        buf.var_type, out.var_type = dt.complex_bf16, dt.complex64
        MX.fft3_mixed(out, buf, graph=graph)

    def between(log):
        got = []
        for group in zip(*[log[i::passes] for i in range(passes)]):
            assert [n for n, _, _ in group] == [str(n) for n in range(passes)]
            assert all(a[2][0] == b[2][1] for a, b in zip(group, group[1:]))  # each reads what the last wrote
            assert group[-1][2][0] == group[0][2][1] + 8
            ((s, y),) = {(s, group[0][2][0]) for _, s, _ in group}
            assert passes == 2 or group[1][2][0] == y + 4 * 256 ** 3 < y + 8 * plan._points
            got.append((s, y))
        return got
    return plan, log, call, between


_Kinds = {"long": _long, "conv": _conv, "mixed": _mixed, "mixed3": lambda m: _mixed(m, 3)}


@pytest.mark.parametrize("kind", ["long", "conv", "mixed", "mixed3"])
def test_recorded_launches_share_nothing_with_calls(device, monkeypatch, kind):
    """Recorded on one stream and submitted on others beside calls on the first; two graphs
    recorded on one stream and submitted on two: each stream its own, kept while a graph
    may run with it."""
    monkeypatch.setattr(scratch, "_streams", {})
    monkeypatch.setattr(scratch, "_pinned", [])
    plan, log, call, between = _Kinds[kind](monkeypatch)
    graphs = [G.CommandGraph(), G.CommandGraph()]
    for g in graphs:
        for b in (1 << 25, 1 << 26):
            call(_Data(b), g)
    assert not log
    for g, s in zip(graphs, (5, 6)):
        g.submit(stream=s)               # captured for s
        assert g._exec_stream == s
    call(_Data(1 << 27), None)
    graphs[0].submit(stream=6, use_graph=False)
    used = {}
    for s, y in between(log):
        used.setdefault(s, set()).add(y)
    assert sorted(used) == [1, 5, 6] and all(len(v) == 1 for v in used.values())
    outside = set.union(*used.values())
    assert len(outside) == 3
    del log[:]
    device.capturing = {7: 9}            # into a capture of the caller's
    for g in graphs:
        g.submit(stream=7)
    device.capturing = {}
    inside = {y for _, y in between(log)}
    assert len(inside) == 2 and not inside & outside
    scratch._streams.clear()
    assert set(device.freed) == used[1]  # the graphs hold theirs
    for g in graphs:
        g.reset()
    assert set(device.freed) == outside  # and captured graphs what they were given
    scratch.clear()
    assert set(device.freed) == outside | inside


def test_a_bound_long_transform_has_its_own_scratch(device):
    plan, log = _long_plan()
    a, b = plan.bind(_Data(100)), plan.bind(_Data(200))
    plan(_Data(300))
    a(1)
    b(1)
    assert len({y for _, y in _between(log)}) == 3


def test_captures_share_nothing(device):
    """With bound launches, calls on any stream, other captures and their own branches."""
    plan, log = _long_plan()

    def used(launch, *a):
        del log[:]
        launch(*a)
        (y,) = {y for _, y in _between(log)}
        return y
    bound = plan.bind(_Data(100))
    outside = {used(bound, 7), used(plan, _Data(200))}
    device.capturing = {1: 11, 2: 11}   # one capture with two branches
    first = [used(plan, _Data(300)) for device.stream in (1, 2)]
    assert [used(plan, _Data(300)) for device.stream in (1, 2)] == first
    device.capturing = {1: 12}          # another on a stream that had one before
    device.stream = 1
    first.append(used(plan, _Data(300)))
    device.capturing = {}
    outside |= {used(plan, _Data(400)) for device.stream in (1, 2, 3, 4)} | {used(bound, 7)}
    assert len(set(first)) == 3 and not outside & set(first)
    for device.capturing in [{1: n} for n in range(20, 60)]:
        device.stream = 1
        used(plan, _Data(300))
    assert len(plan._captured) == LG.SCRATCH_CAPTURES and not set(device.freed) & set(first)


def test_two_threads_convolve_in_turn(device, monkeypatch):
    monkeypatch.setattr(scratch, "_streams", {})
    plan, log, call, between = _conv(monkeypatch)
    inside, other = threading.Event(), threading.Event()

    class Slow(_Kernel):
        def launch_raw(self, ptrs, consts=b"", stream=None):
            super().launch_raw(ptrs, consts, stream)
            if not inside.is_set():
                inside.set()
                other.wait(0.3)
    plan.kernels_[0] = Slow(log, "rows")
    t = threading.Thread(target=lambda: (inside.wait(), call(_Data(1 << 26), None), other.set()))
    t.start()
    call(_Data(1 << 25), None)
    t.join()
    between(log)
    assert [p[0] for _, _, p in log] == [1 << 25] * 3 + [1 << 26] * 3


def test_two_threads_on_one_stream_take_turns(device):
    """The second thread calls while the first is between its launches; on the stream of each
    thread (one handle, hipStreamPerThread) they have different scratch."""
    for stream, apart in ((1, False), (2, True)):
        device.stream = stream
        plan, log = _long_plan()
        inside, other = threading.Event(), threading.Event()

        class Slow(_Kernel):
            def launch_raw(self, ptrs, consts=b"", stream=None):
                super().launch_raw(ptrs, consts, stream)
                if not inside.is_set():
                    inside.set()
                    other.wait(0.3)    # as long as the other thread would need
        rows = plan.kernels[1][1]
        plan.kernels = {c: (Slow(log, "cols"), rows) for c in (1, 2)}

        def second():
            inside.wait()
            plan(_Data(1 << 30))
            other.set()
        t = threading.Thread(target=second)
        t.start()
        plan(_Data(1 << 25))
        t.join()
        if not apart:
            _between(log)              # whole pairs,
            x = [p[1] if k == "cols" else p[0] for k, _, p in log]
            assert len(log) == 8 and [v < 1 << 29 for v in x] in ([True] * 4 + [False] * 4, [False] * 4 + [True] * 4)
        else:
            y = {(p[1] if k == "cols" else p[0]) < 1 << 29: p[0] if k == "cols" else p[1] for k, _, p in log}
            assert len(set(y.values())) == 2


def test_plans_on_one_stream_share_a_buffer(device, monkeypatch):
    """What calls keep grows with the largest plan and the streams, not with the plans."""
    monkeypatch.setattr(scratch, "_streams", {})
    plans = []
    for points in (64, 32, 128, 64):
        plan, log = _long_plan(points)
        plan._init_scratch(points)
        plans.append((plan, log))
        plan(_Data(100))
    got = [_between(log)[0][1] for _, log in plans]
    assert got[0] == got[1] and got[2] == got[3] != got[0]  # the third needs more
    assert device.freed == [got[0]] and len(scratch._streams) == 1
    for device.stream in range(20):
        plans[0][0](_Data(100))
    assert len(scratch._streams) == scratch.SCRATCH_STREAMS
    monkeypatch.setattr(scratch, "_pinned", [])
    scratch.clear()
    assert not scratch._streams and len(device.freed) == 21


def test_lengths_of_the_ragged_executor(device, monkeypatch):
    """Prime factors above 13: a plan for each stream's calls and for each graph, whose launches
    share it; a capture, which cannot build one, takes the newest."""
    from vkdispatch_amd.fft import ragged
    made, ran = [], []

    class Plan:
        n_items = 3

        def __init__(self, sizes, **kw):
            assert sizes == [20011] * 3
            made.append(self)

        def bind(self, buf):
            return lambda stream=None: ran.append((self, device.stream if stream is None else stream))

        def __call__(self, buf):
            self.bind(buf)()
    monkeypatch.setattr(ragged, "RaggedFFT", Plan)
    monkeypatch.setattr(F, "_RAGGED_PLANS", {})
    monkeypatch.setattr(scratch, "_pinned", [])

    def call(graph=None):
        assert F._large_or_prime_fallback((_Data(100),), (3, 20011), None, False, True, False, None, None, dt.complex64,
                                          dt.complex64, None, graph)
    for device.stream in (1, 5, 1):
        call()
    device.stream = 1
    graphs = [G.CommandGraph(), G.CommandGraph()]
    for g in graphs:
        call(g)
        call(g)
    assert len(made) == 4
    for g, s in zip(graphs, (7, 8)):
        g._replay(s)
    owners = {}
    for plan, s in ran:
        owners.setdefault(s, set()).add(plan)
    assert sorted(owners) == [1, 5, 7, 8] and all(len(p) == 1 for p in owners.values())
    assert len(set.union(*owners.values())) == 4
    device.stream, device.capturing = 9, {9: 1}
    call()
    assert len(made) == 4 and ran[-1] == (made[0], 9)  # stream 1 called last
    graphs[0].submit(stream=9)
    assert scratch._pinned == [made[0], made[2]]  # what was captured is kept,
    device.capturing = {}
    for device.stream in range(20, 30):
        call()
    (calls,) = F._RAGGED_PLANS.values()
    assert len(calls) == scratch.SCRATCH_STREAMS and made[0] not in calls.values()  # also when no call has it any more


def test_a_graph_waits_for_a_call_to_be_enqueued(device, monkeypatch):
    """A thread submits a graph on the stream of a call that is between its launches."""
    monkeypatch.setattr(scratch, "_streams", {})
    plan, log, call, _ = _long(monkeypatch)
    graph = G.CommandGraph()
    call(_Data(1 << 25), graph)
    graph.capture(1)
    del log[:]
    device.vkx_graph_launch = lambda ex, s: log.append(("graph", s, ())) or 0
    inside, other = threading.Event(), threading.Event()

    class Slow(_Kernel):
        def launch_raw(self, ptrs, consts=b"", stream=None):
            super().launch_raw(ptrs, consts, stream)
            if not inside.is_set():
                inside.set()
                other.wait(0.3)
    plan.kernels = {c: (Slow(log, "cols"), plan.kernels[c][1]) for c in (1, 2)}
    t = threading.Thread(target=lambda: (inside.wait(), graph.submit(stream=1), other.set()))
    t.start()
    call(_Data(1 << 26), None)
    t.join()
    assert [n for n, _, _ in log] in (["cols", "rows"] * 2 + ["graph"], ["graph"] + ["cols", "rows"] * 2)
