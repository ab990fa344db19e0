"""Plans of the one-workgroup 2-D convolution (fft/half2d.py) on the CPU."""
import numpy as np
import pytest

import vkdispatch_amd as vd
from vkdispatch_amd.fft import fused, half2d
from vkdispatch_amd.fft.planner import LDS_BYTES_MAX, slots


@pytest.mark.parametrize("h", [2, 3, 13, 32, 60, 97, 128, 210, 512])
@pytest.mark.parametrize("m", [2, 3, 16, 49, 64, 105, 256])
def test_whole_plan_fits(h, m):
    plan = half2d.whole_plan(h, m)
    if plan is None:
        assert h == 97 or h * m * 8 > LDS_BYTES_MAX - 8 * (2 * (h + m) + m)
        return
    (rr, rtt), (cr, ctt), pitch = plan
    assert np.prod(rr) == m and np.prod(cr) == h and pitch >= m
    for n, radices, tt in ((m, rr, rtt), (h, cr, ctt)):
        assert 1 <= tt <= 64 and max(slots(n, r, tt) for r in radices) <= 20
    # the image, the twiddles of rows (m - 1) and of columns both ways, and the roots
    assert 8 * (h * pitch + (m - 1) + 2 * (h - 1) + m // 2 + 1) <= LDS_BYTES_MAX


def test_roots_hold_every_twiddle():
    """A pass of radix R after NS points takes W_(R NS)^(r k): roots of order lcm(2m, h) at
    multiples of lcm / (R NS), an integer for every prefix of either radix list."""
    for h, m in ((60, 50), (210, 49), (128, 64), (13, 3)):
        (rr, _), (cr, _), _ = half2d.whole_plan(h, m)
        order = np.lcm(2 * m, h)
        for radices in (rr, cr, cr[::-1]):
            assert all(order % int(np.prod(radices[:i + 1])) == 0 for i in range(len(radices)))


def test_which_convolutions_take_one_launch():
    def path(shape, **kw):
        return type(fused.plan_for_shape(shape, **kw)).__name__
    assert path((256, 128, 128), kernel_inner_only=True) == "HalfWhole"
    assert path((4, 64, 64), kernel_inner_only=True) == "HalfWhole"
    assert path((4, 64, 64)) == "HalfWhole"                                     # a kernel per image
    assert path((64, 128, 128), kernel_inner_only=True) == "NoneType"           # too few of this size
    assert path((256, 200, 200), kernel_inner_only=True) == "NoneType"          # too large
    assert path((4, 64, 63), kernel_inner_only=True) == "NoneType"              # odd width
    assert path((4, 64, 64), kernel_inner_only=True, transposed_kernel=True) == "NoneType"
    assert path((4, 64, 64), kernel_inner_only=True, compute_type=vd.complex128) == "NoneType"
    assert path((4, 512, 512), kernel_inner_only=True) == "Conv2DPhases"
