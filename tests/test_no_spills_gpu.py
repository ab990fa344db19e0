"""GPU parity of strided kernels whose first plan spills (tests/test_no_spills.py): rel-L2 5e-6 against
FP64, complex128 1e-13."""
import numpy as np
import pytest

import oracle as O
import vkdispatch_amd as vd
import vkdispatch_amd.codegen as vc
from tests._gpu_common import assert_close, crand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,s", [(468, 64), (468, 65), (2916, 16)])
def test_transforms_in_double(n, s):
    data = crand(np.random.default_rng(n), (2, n, s), np.complex128)
    buf = vd.asbuffer(data)
    for inverse in (False, True):
        buf.write(data)
        vd.fft.fft(buf, axis=1, inverse=inverse, compute_type=vd.complex128)
        assert_close(buf.read(0), O.fft_axis(data, 1, inverse=inverse), rel=1e-13)


@pytest.mark.parametrize("n,s", [(1000, 320), (1125, 64), (2304, 33)])
def test_a_kernel_per_batch(n, s):
    rng = np.random.default_rng(n)
    data, kern = crand(rng, (2, n, s)), crand(rng, (2, n, s))
    buf, kbuf = vd.asbuffer(data), vd.asbuffer(kern)
    vd.fft.convolve(buf, kbuf, axis=1)
    assert_close(buf.read(0), O.convolve_axis(data, kern, 1))


@pytest.mark.parametrize("n,s,num", [(882, 513, 2), (1000, 64, 3), (2048, 64, 2), (490, 321, 3)])
def test_several_kernels(n, s, num):
    rng = np.random.default_rng(n + num)
    data = crand(rng, (2, n, s))
    kern = [crand(rng, (2, n, s)) for _ in range(num)]
    buf, kbuf = vd.asbuffer(data), vd.asbuffer(np.concatenate(kern))
    out = vd.Buffer((2 * num, n, s), vd.complex64)

    @vd.map
    def kmap(k: vc.Buffer[vd.complex64]):
        op = vd.fft.read_op()
        kv = vc.new_register(vd.complex64)
        op.read_from_buffer(k, register=kv, io_index=op.io_index + vd.fft.mapped_kernel_index() * 2 * n * s)
        op.register[:] = vc.mult_complex(op.register, kv.conjugate())

    @vd.map
    def omap(o: vc.Buffer[vd.complex64]):
        op = vd.fft.write_op()
        op.write_to_buffer(o, io_index=op.io_index + vd.fft.mapped_kernel_index() * 2 * n * s)

    vd.fft.convolve(out, buf, kbuf, kernel_map=kmap, kernel_num=num, output_map=omap, axis=1, buffer_shape=(2, n, s))
    got = out.read(0)
    for i, k in enumerate(kern):
        assert_close(got[2 * i:2 * i + 2], O.convolve_axis(data, k, 1))
