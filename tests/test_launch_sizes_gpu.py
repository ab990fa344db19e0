"""GPU parity of plans that depend on the size of a launch: few rows on both sides of the line, narrow
tiles.  rel-L2 5e-6 against FP64, complex128 1e-13."""
import numpy as np
import pytest

import oracle as O
import vkdispatch_amd as vd
from tests._gpu_common import assert_close, crand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 45), (5, 143), (3, 500), (1048, 500), (1049, 500), (7, 1001), (2, 2187), (61, 338),
                                   (1, 4000)], ids=str)
def test_rows(shape):
    data = crand(np.random.default_rng(1), shape)
    buf = vd.asbuffer(data)
    for inverse in (False, True):
        buf.write(data)
        vd.fft.fft(buf, inverse=inverse)
        assert_close(buf.read(0), O.fft_axis(data, 1, inverse=inverse))
    kern = crand(np.random.default_rng(2), shape[1:])
    buf.write(data)
    vd.fft.convolve(buf, vd.asbuffer(kern), axis=1, kernel_inner_only=True)
    assert_close(buf.read(0), O.convolve_axis(data, kern, 1, kernel_inner_only=True))


@pytest.mark.parametrize("shape", [(1, 90), (5, 286), (3, 1000), (524, 1000), (525, 2000), (7, 2002), (2, 4374), (61, 676)], ids=str)
def test_real_rows(shape):
    data = np.random.default_rng(3).random(shape).astype(np.float32)
    buf = vd.asrfftbuffer(data)
    vd.fft.rfft(buf)
    assert_close(buf.read_fourier(0), np.fft.rfft(data.astype(np.float64)))
    vd.fft.irfft(buf)
    assert_close(buf.read_real(0), data)


@pytest.mark.parametrize("shape", [(1, 125, 32), (2, 1000, 65), (2, 512, 257), (1, 972, 33), (4, 1000, 257), (3, 338, 50),
                                   (17, 243, 65), (2, 2000, 40)], ids=str)
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
def test_columns(shape, dtype):
    t, rel = (vd.complex64, 5e-6) if dtype == "complex64" else (vd.complex128, 1e-13)
    rng = np.random.default_rng(4)
    data, kern = crand(rng, shape, np.dtype(dtype)), crand(rng, shape[1:], np.dtype(dtype))
    guard = np.full(64, 7 - 3j, data.dtype)   # what follows the buffer's last element stays as it is
    whole = np.concatenate([data.ravel(), guard])
    buf = vd.Buffer((whole.size,), t)
    for inverse in (False, True):
        buf.write(whole)
        vd.fft.fft(buf, buffer_shape=shape, axis=1, inverse=inverse, compute_type=t)
        got = buf.read(0)
        assert_close(got[:data.size].reshape(shape), O.fft_axis(data, 1, inverse=inverse), rel=rel)
        assert (got[data.size:] == guard).all()
    buf.write(whole)
    kbuf = vd.Buffer(kern.shape, t)
    kbuf.write(kern)
    vd.fft.convolve(buf, kbuf, buffer_shape=shape, axis=1, kernel_inner_only=True, compute_type=t)
    got = buf.read(0)
    assert_close(got[:data.size].reshape(shape), O.convolve_axis(data, kern, 1, kernel_inner_only=True), rel=rel)
    assert (got[data.size:] == guard).all()
