"""Strided plans of many values a thread on the CPU: what needs more registers than there are has
a plan that compiles without spills (gfx950 code objects)."""
import pytest

import vkdispatch_amd as vd
import vkdispatch_amd.codegen as vc
from vkdispatch_amd.fft import planner as P
from vkdispatch_amd.fft.kernels import SpillError, check_no_spill
from vkdispatch_amd.fft.shader_factories import make_convolution_shader, make_fft_shader

C64, C128 = vd.complex64, vd.complex128


def _maps(t):
    @vd.map
    def kmap(kbuf: vc.Buffer[t]):
        op = vd.fft.read_op()
        k = vc.new_register(t)
        op.read_from_buffer(kbuf, register=k, io_index=op.io_index + (vd.fft.mapped_kernel_index() or 0) * 4096)
        op.register[:] = vc.mult_complex(op.register, k.conjugate())

    @vd.map
    def omap(obuf: vc.Buffer[t]):
        op = vd.fft.write_op()
        op.write_to_buffer(obuf, io_index=op.io_index + (vd.fft.mapped_kernel_index() or 0) * 4096)
    return kmap, omap


@pytest.mark.parametrize("shape,t,num,hooked", [
    ((8, 882, 513), C64, 2, False), ((8, 2048, 513), C64, 2, True), ((8, 1152, 513), C64, 2, True),
    ((8, 490, 320), C64, 3, False), ((8, 1000, 320), C64, 3, False), ((8, 1024, 320), C64, 3, False),
    ((8, 700, 320), C128, 2, False), ((8, 864, 320), C128, 2, False), ((3, 1000, 320), C128, 3, False),
    ((8, 1000, 320), C64, 1, False), ((8, 1125, 320), C64, 1, False), ((8, 2304, 320), C64, 1, False),
    ((8, 468, 320), C128, 1, False), ((8, 1000, 512), C64, 1, True), ((8, 900, 512), C128, 1, True),
    ((8, 341, 64), C128, 2, False), ((8, 4032, 320), C64, 2, False)], ids=str)
def test_convolutions(shape, t, num, hooked):
    kmap, omap = _maps(t) if hooked else (None, None)
    k = make_convolution_shader(shape, kmap, num, 1, output_map=omap, input_type=t, output_type=t, kernel_type=t,
                                compute_type=t)
    check_no_spill(k)


@pytest.mark.parametrize("n", [468, 2916])
@pytest.mark.parametrize("s", [64, 321])
def test_transforms(n, s):
    check_no_spill(make_fft_shader((8, n, s), 1, input_type=C128, output_type=C128, compute_type=C128))


def test_a_roomier_plan_keeps_what_its_kernel_needs():
    """The LDS row of a real transform, and a grid that covers the batch."""
    g = P.AxisGeometry((40, 2400), 1, 2400, 1, 40)
    for p in P.roomier_plans(g, "float", "rfft", need_lds=True):
        assert p.LDS_ELEMS >= p.B * p.NP and p.NWG * p.B >= 40
    g = P.AxisGeometry.of((40, 1000, 320), 1)
    plans = list(P.roomier_plans(g, "float", "conv"))
    assert len(plans) == 2 and all(p.VMAX < P.make_plan(g, kind="conv").VMAX and p.NWG_INNER * p.B >= 320 for p in plans)


def test_nothing_is_compiled_before_it_is_wanted(monkeypatch):
    """Plans are made without compiling; a kernel that spills is replaced whole, once."""
    from vkdispatch_amd.fft import kernels as K
    compiled = []
    compile_source = K.compile_source
    monkeypatch.setattr(K, "compile_source", lambda s: compiled.append(s) or compile_source(s))
    vd.fft.cache_clear()
    fine, spills = make_fft_shader((8, 600, 320), 1), make_convolution_shader((8, 1000, 320), None, 1, 1)
    assert not compiled
    first = spills._plan
    check_no_spill(fine)
    check_no_spill(spills)
    assert spills.plan != first and spills.plan.VMAX < first.VMAX
    meta = K.parse_launch_comment(spills.source)
    assert meta == spills.launch_metadata() and meta["radices_fwd"] == list(spills.plan.radices)
    assert meta["grid"] == list(spills.plan.grid) and meta["block"][0] == spills.plan.BLOCK
    n = len(compiled)
    spills.settle()
    assert len(compiled) == n


def test_an_override_is_not_replaced():
    """The autotuner times the plan it asked for, or learns that it spills."""
    g = P.AxisGeometry.of((8, 1000, 320), 1)
    p = P.make_plan(g, kind="conv")
    P.set_override(g, "float", "conv", p.radices, p.TT, p.B)
    try:
        vd.fft.cache_clear()
        with pytest.raises(SpillError):
            check_no_spill(make_convolution_shader((8, 1000, 320), None, 1, 1))
    finally:
        P.set_override(g, "float", "conv")
        vd.fft.cache_clear()
