"""Plans that depend on how much a launch has to do (fft/planner.py), on the CPU."""
import numpy as np
import pytest

from vkdispatch_amd.fft import planner as P

LENGTHS = [36, 45, 60, 96, 125, 143, 243, 338, 480, 500, 686, 720, 972, 1000, 1001, 1250, 2000, 2187, 4000]


@pytest.mark.parametrize("real,elem", [("float", 8), ("double", 16)])
@pytest.mark.parametrize("kind", ["fft", "conv", "rfft"])
def test_plans_fit_at_every_size(real, elem, kind):
    for n in LENGTHS:
        for s in ((1,) if kind == "rfft" else (1, 32, 65, 257, 320)):
            for outer in (1, 2, 17, 300, 5000):
                try:
                    p = P.make_plan(P.AxisGeometry((outer, n, s), 1, n, s, outer), real, kind=kind,
                                    need_lds=kind == "rfft")
                except ValueError:
                    assert P.radix_plan(n)[1] > P.MAX_THREADS or n * elem > 128 * 1024
                    continue
                assert np.prod(p.radices) == n and p.BLOCK <= P.MAX_THREADS and p.lds_bytes <= P.LDS_BYTES_MAX
                assert all(p.TT * -(-(n // r) // p.TT) >= n // r for r in p.radices)
                assert p.NWG_INNER * p.B >= s if s > 1 else p.NWG * p.B >= outer
                if kind == "rfft":
                    assert p.LDS_ELEMS >= p.B * p.NP
                if p.LPW:
                    assert p.LPW * p.TT <= 64 and p.BLOCK // 64 * p.LPW == p.B


def test_few_rows_and_many():
    """Up to FEW_POINTS a row takes more threads and a workgroup one wave; complex128 and powers
    of two are as they were."""
    def rows(outer, n, real="float"):
        return P.make_plan(P.AxisGeometry((outer, n), 1, n, 1, outer), real)
    few, many = rows(P.FEW_POINTS // 500, 500), rows(P.FEW_POINTS // 500 + 1, 500)
    assert few.VMAX <= 10 < many.VMAX and few.BLOCK == 64 < many.BLOCK
    assert rows(1, 500, "double").radices == rows(5000, 500, "double").radices
    assert rows(1, 512).radices == rows(5000, 512).radices


def test_few_tiles_and_many():
    """Whole lines where the launch fills the chip several times over; narrower tiles where
    it does not, or where the last round of large workgroups would be nearly empty."""
    def cols(outer, n, s):
        return P.make_plan(P.AxisGeometry.of((outer, n, s), 1), kind="conv")
    assert cols(40, 1000, 257).B == 16 and cols(40, 1000, 320).B == 16
    assert cols(2, 1000, 257).B < 16 and cols(16, 1000, 257).B < 16
    assert cols(16, 1000, 257).NWG <= 256 * (P.LDS_BYTES_MAX // cols(16, 1000, 257).lds_bytes)
    assert cols(40, 1000, 24).radices == cols(500, 1000, 24).radices  # strides it says nothing about


def test_which_batches_of_small_images_take_one_launch():
    """Beyond two images to a CU, only sizes whose workgroups keep it busy."""
    from vkdispatch_amd.fft import half2d
    def pays(n, h, w):
        return half2d.whole_pays(n, h, w // 2)
    assert all(pays(n, h, w) for n in (96, 256, 512) for h, w in ((96, 96), (128, 128), (60, 100), (200, 100)))
    assert all(pays(n, h, w) for n in (600, 1024) for h, w in ((32, 32), (48, 96), (64, 128), (128, 128), (16, 1000)))
    assert not any(pays(n, h, w) for n in (800, 1024) for h, w in ((96, 96), (60, 100), (96, 120), (128, 96)))
    assert not pays(95, 128, 128) and pays(1, 64, 64) and not pays(1024, 160, 200)
