"""GPU parity of the single-launch plans: wave-owned rows with idle lanes, one long row per
workgroup, strided columns of whole lines, padded exchanges and grids with idle workgroups.
Bounds: the FP64 oracle at the suite's rel-L2 5e-6; complex128 1e-13 (5 passes of a few eps)."""
import numpy as np
import pytest

import oracle as O
import vkdispatch_amd as vd
from tests._gpu_common import assert_close, crand

pytestmark = pytest.mark.gpu

ROWS = [(1, 33), (5, 33), (70, 45), (33, 60), (129, 96), (17, 243), (41, 600), (3, 961), (23, 1500), (2, 2160), (9, 2187),
        (1, 9282), (2, 10000)]
COLUMNS = [(1, 34, 3), (2, 600, 37), (3, 1000, 21), (1, 1000, 64), (40, 60, 33), (17, 96, 50), (9, 512, 65), (2, 1024, 129),
           (1, 4096, 11), (30, 100, 321), (5, 720, 16), (3, 961, 18)]


@pytest.mark.parametrize("shape", ROWS + COLUMNS, ids=str)
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
def test_transform(shape, dtype):
    t, rel = (vd.complex64, 5e-6) if dtype == "complex64" else (vd.complex128, 1e-13)
    if dtype == "complex128" and (max(shape[1], 1) > 8192):
        pytest.skip("needs more LDS than a workgroup has")
    data = crand(np.random.default_rng(5), shape, np.dtype(dtype))
    guard = 64   # words after the buffer's last element stay as they are
    whole = np.concatenate([data.ravel(), np.full(guard, 7 - 3j, data.dtype)])
    buf = vd.Buffer((whole.size,), t)
    for inverse in (False, True):
        buf.write(whole)
        vd.fft.fft(buf, buffer_shape=shape, axis=1, inverse=inverse, compute_type=t)
        got = buf.read(0)
        assert_close(got[:data.size].reshape(shape), O.fft_axis(data, 1, inverse=inverse), rel=rel)
        assert (got[data.size:] == whole[data.size:]).all()


@pytest.mark.parametrize("shape", [(5, 66), (70, 90), (33, 120), (41, 1200), (2, 4320), (9, 486)], ids=str)
def test_real_rows(shape):
    data = np.random.default_rng(6).random(shape).astype(np.float32)
    buf = vd.asrfftbuffer(data)
    vd.fft.rfft(buf)
    assert_close(buf.read_fourier(0), np.fft.rfft(data.astype(np.float64)))
    vd.fft.irfft(buf)
    assert_close(buf.read_real(0), data)


@pytest.mark.parametrize("shape", [(33, 60), (9, 600), (2, 2160), (40, 60, 33), (3, 1000, 21), (30, 100, 65)], ids=str)
@pytest.mark.parametrize("how", ["each", "inner", "transposed", "transposed inner"])
def test_convolution(shape, how):
    rng = np.random.default_rng(7)
    inner = "inner" in how
    data, kern = crand(rng, shape), crand(rng, shape[1:] if inner else shape)
    buf, kbuf = vd.asbuffer(data), vd.asbuffer(kern)
    if "transposed" in how:
        size = vd.fft.get_transposed_size(shape, axis=1)
        out = vd.Buffer((size,), vd.complex64)
        vd.fft.transpose(kbuf, conv_shape=shape, out_buffer=out, axis=1, kernel_inner_only=inner)
        kbuf = out
    vd.fft.convolve(buf, kbuf, axis=1, transposed_kernel="transposed" in how, kernel_inner_only=inner)
    assert_close(buf.read(0), O.convolve_axis(data, kern, 1, kernel_inner_only=inner))


def test_signal_range_with_idle_lanes():
    shape = (70, 90)
    data = crand(np.random.default_rng(8), shape)
    buf = vd.asbuffer(data)
    vd.fft.fft(buf, axis=1, input_signal_range=(0, 41))
    part = data.copy()
    part[:, 41:] = 0
    assert_close(buf.read(0), O.fft_axis(part, 1))


@pytest.mark.parametrize("shape", [(1, 640, 32), (3, 500, 16), (70, 96, 64), (65, 200, 64), (26, 540, 160), (70, 90, 32)], ids=str)
def test_kernels_scheduled_for_fewer_waves(shape):
    """Full tiles of many values a thread: launches that leave CUs idle, and others."""
    test_convolution(shape, "inner")
    test_transform((shape[0], shape[1], shape[2]), "complex64")
    test_transform((shape[0], shape[1], shape[2]), "complex128")
