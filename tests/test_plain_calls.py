"""Calls without maps find their kernel by what decides it: the same kernel and the same
refusals as with every step resolved anew (CPU, dispatches recorded)."""
import pytest

import vkdispatch_amd as vd
from vkdispatch_amd.fft import functions as F


def _fake(shape, vt=vd.complex64):
    return vd.Buffer(shape, vt, external=(0x10000000, None, True))


@pytest.fixture
def calls(monkeypatch):
    got = []
    monkeypatch.setattr(F, "dispatch", lambda kernel, values, graph=None: got.append((kernel.source, values, graph)))
    return got


def _general(monkeypatch):
    monkeypatch.setattr(F, "_plain_fft", lambda *a: (None, 0))
    monkeypatch.setattr(F, "_plain_convolution", lambda *a: (None, float("inf")))


FFT_CALLS = [dict(), dict(axis=0), dict(axis=1, inverse=True), dict(inverse=True, normalize_inverse=False),
             dict(input_signal_range=(0, 9)), dict(compute_type=vd.complex128), dict(buffer_shape=(3, 10)),
             dict(buffer_shape=[3, 10]), dict(axis=7), dict(input_type=vd.complex128), dict(output_type=vd.float32),
             dict(buffer_shape=(30, 400)), dict(input_signal_range=(9, 3)), dict(r2c=True, axis=0)]
CONV_CALLS = [dict(), dict(axis=0), dict(kernel_inner_only=True), dict(normalize=False), dict(kernel_num=2),
              dict(transposed_kernel=True), dict(kernel_type=vd.complex32), dict(compute_type=vd.complex128),
              dict(kernel_num=0), dict(axis=5), dict(input_type=vd.complex32), dict(buffer_shape=(6, 30, 20))]


def _outcome(fn, calls):
    calls.clear()
    try:
        fn()
        return list(calls)
    except Exception as e:  # the refusal's type and words
        return type(e), str(e)


@pytest.mark.parametrize("vt", [vd.complex64, vd.complex32, vd.complex128, vd.float32])
def test_same_kernel_or_refusal(vt, calls, monkeypatch):
    b, k, small = _fake((6, 30, 20), vt), _fake((6, 30, 20)), _fake((20,))
    todo = [lambda kw=kw: F.fft(b, **kw) for kw in FFT_CALLS]
    todo += [lambda kw=kw, q=q: F.convolve(b, q, **kw) for kw in CONV_CALLS for q in (k, small)]
    todo += [lambda: F.fft(b, k), lambda: F.fft(small, buffer_shape=(40,)), lambda: F.convolve(b, k, small)]
    kept = [_outcome(fn, calls) for _ in range(2) for fn in todo]
    _general(monkeypatch)
    assert kept == [_outcome(fn, calls) for fn in todo] * 2


def test_cache_info_counts_and_clears(calls):
    vd.fft.cache_clear()
    b = _fake((6, 30, 20))
    for _ in range(3):
        F.fft(b)
    assert vd.fft.get_cache_info().hits == 2 and vd.fft.get_cache_info().misses == 1
    vd.fft.cache_clear()
    F.fft(b)
    assert vd.fft.get_cache_info().hits == 0 and vd.fft.get_cache_info().misses == 1
