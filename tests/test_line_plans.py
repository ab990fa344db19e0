"""Plans of single-launch transforms (fft/planner.py) on the CPU: rows whose waves hold whole
transforms, strided columns of whole lines, and what neither may change."""
import numpy as np
import pytest

import vkdispatch_amd as vd
from vkdispatch_amd.fft import planner as P
from vkdispatch_amd.fft.shader_factories import make_convolution_shader, make_fft_shader

LENGTHS = [33, 34, 40, 60, 96, 100, 162, 243, 480, 600, 961, 1000, 1024, 1155, 2048, 2160, 4096, 8192, 9282, 10000,
           13122, 14406, 16384]


def _plan(n, s, real, **kw):
    return P.make_plan(P.AxisGeometry((40, n, s), 1, n, s, 40), real, **kw)


@pytest.mark.parametrize("real,elem", [("float", 8), ("double", 16)])
@pytest.mark.parametrize("s", [1, 3, 16, 321])
def test_plans_fit_and_cover_every_butterfly(real, elem, s):
    for n in LENGTHS:
        try:
            p = _plan(n, s, real)
        except ValueError:
            assert n * elem > 128 * 1024 or P.radix_plan(n)[1] > P.MAX_THREADS  # refused as ever
            continue
        assert np.prod(p.radices) == n and p.BLOCK <= P.MAX_THREADS and p.lds_bytes <= P.LDS_BYTES_MAX
        assert all(P.slots(n, r, p.TT) * r <= p.VMAX or P.slots(n, r, p.TT) <= p.VMAX for r in p.radices)
        if p.LPW:   # the lanes of a wave hold whole transforms, those of all waves the workgroup's
            assert s == 1 and p.WAVE_LOCAL and p.LPW * p.TT <= 64 and p.BLOCK // 64 * p.LPW == p.B
        assert p.NWG_INNER * p.B >= s if s > 1 else p.NWG * p.B >= 40


@pytest.mark.parametrize("n,s,real", [(512, 64, "float"), (600, 401, "float"), (1000, 320, "float"),
                                      (720, 64, "double"), (1000, 24, "float")])
def test_padded_addresses_are_distinct_and_inside(n, s, real):
    """lds_addr of every (position, transform) of a padded plan, and its legs' constant steps."""
    p = _plan(n, s, real)
    assert p.CPAD
    r0 = p.radices[0]
    addr = np.array([[pos * p.B + b + pos // r0 * p.B for b in range(p.B)] for pos in range(n)])
    assert len(np.unique(addr)) == addr.size and addr.max() < p.LDS_ELEMS
    for r, ns in p.fwd:     # the steps that the kernel takes as constants
        w = n // r
        if w % r0 == 0:
            assert (addr[np.arange(w) + w, 0] - addr[:w, 0] == (w + w // r0) * p.B).all()
        if ns % r0 == 0:
            base = np.array([(j // ns) * ns * r + j % ns for j in range(w)])
            assert (addr[base + ns, 0] - addr[base, 0] == (ns + ns // r0) * p.B).all()


@pytest.mark.parametrize("nwg", [1, 15, 16, 17, 24, 41])
def test_idle_workgroups_fill_the_grid_to_whole_xcds(nwg):
    p = P.make_plan(P.AxisGeometry((nwg, 64, 16), 1, 64, 16, nwg))
    assert p.NWG == nwg
    assert P.whole_xcds(p).NWG == (nwg if nwg < 16 else -(-nwg // 8) * 8)


@pytest.mark.parametrize("shape,axis,size", [((4, 64, 33), 1, 12288), ((7, 600), 1, 7680), ((3, 1000, 21), 1, 75000),
                                             ((5, 60), 1, 320), ((40, 96, 15), 1, 76800)])
def test_transposed_layout_is_what_it_was(shape, axis, size):
    """A stored transposed kernel's order follows from threads, radices and B: radix_plan's."""
    assert vd.fft.get_transposed_size(shape, axis=axis) == size
    k = vd.fft.make_convolution_shader(shape, None, 1, axis, transposed_kernel=True)
    t = vd.fft.make_transpose_shader(shape, axis)
    assert list(k.plan.radices) == P.radix_plan(shape[axis])[0] and k.plan.TT == P.radix_plan(shape[axis])[1]
    assert (k.plan.B, k.plan.NWG, k.plan.LPW) == (t.plan.B, t.plan.NWG, 0)


@pytest.mark.parametrize("shape,real,conv,want", [
    ((1, 640, 320), "float", True, (1, 2)), ((1, 640, 320), "float", False, (1, 2)),    # few workgroups
    ((26, 500, 320), "float", True, (2, 3)), ((65, 200, 320), "float", True, (1, 3)),
    ((26, 500, 320), "float", False, None), ((32, 400, 320), "float", True, None),      # measured slower
    ((20, 640, 320), "float", True, None),                                              # 8 waves a workgroup
    ((26, 500, 257), "float", True, None), ((64, 512, 1), "float", True, None),         # part tiles, rows
    ((40, 160, 320), "double", False, (1, 3)), ((72, 90, 320), "double", False, (1, 3)),
    ((40, 160, 320), "double", True, None)])
def test_waves_to_schedule_for(shape, real, conv, want):
    """The bound holds the workgroup's own waves, and what it gives the compiler spills nothing."""
    plan = P.make_plan(P.AxisGeometry.of(shape, 1), real, kind="conv" if conv else "fft")
    got = P.wave_bounds(plan, conv)
    assert got == want
    if got is None:
        return
    assert got[0] <= got[1] and 4 * P.WAVE * got[0] >= plan.BLOCK
    c = vd.complex64 if real == "float" else vd.complex128
    k = make_convolution_shader(shape, None, 1, 1, kernel_inner_only=True) if conv else \
        make_fft_shader(shape, 1, input_type=c, output_type=c, compute_type=c)
    assert f"amdgpu_waves_per_eu({got[0]}, {got[1]})" in k.source
    assert k.code_object_info()["private_bytes"] == 0
