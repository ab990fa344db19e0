"""Column kernels over packed half spectra (``csrc/device/vkx_half.h``): the middle of 2-D
real convolutions and of their adjoint, between the row kernels that write and read such
spectra (``make_real_rows_shader(..., packed=True)``)."""
from __future__ import annotations

import math
from functools import lru_cache
from typing import Optional, Tuple

import numpy as np

from .. import dtypes as dt
from .hooks import Arg
from .kernels import CompiledKernel, kernel_symbol, translation_unit
from .long import TilePlan, tile_radices
from .planner import LDS_BYTES_MAX, MAX_THREADS, KernelPlan, groupings, pass_list, slots
from .precision import kernel_real_type

LDS_SHARED = 80 * 1024  # two workgroups on a CU
SLOTS = 512             # two workgroups on each CU
WHOLE_WAVES = 16        # most waves of a workgroup that holds an image
WHOLE_LDS = 100 * 1024  # and the most of its LDS


def column_tile(h: int, elem: int) -> Optional[TilePlan]:
    """Tile of h-point columns, or None.  Two workgroups on a CU matter more than the width
    of a tile: 1024 points, 32 images of 512 columns, 8 columns (76 KB of LDS) 60 us, 16
    (one workgroup) 66 us; below that 16, whole 128-byte lines."""
    hit = tile_radices(h, 32 if elem == 8 else 16)
    if hit is None:
        return None
    radices, tt, _ = hit
    fits = [t for t in (TilePlan(h, radices, tt, b, False) for b in (16, 8, 4))
            if (t.lds_elems + h) * elem <= LDS_BYTES_MAX and tt * t.B <= MAX_THREADS]
    for t in fits:
        if (t.lds_elems + h) * elem <= LDS_SHARED and t.TT * t.B <= 512:
            return t
    return fits[0] if fits else None


def _images_per_workgroup(images: int, tiles: int) -> int:
    """As many as leave two rounds of workgroups, up to 4: K then stays in registers over
    them (4 images 60 us, 2 60.5, 1 75), and a round that is not full costs little."""
    per = 4
    while per > 1 and tiles * -(-images // per) < 2 * SLOTS:
        per //= 2
    return per


def _column_kernel(kind: str, body: str, h: int, m: int, images: int, ctype, extra_tiles: int, conj: bool,
                   slots_used: int, tag: str, keep: bool = False) -> CompiledKernel:
    real = kernel_real_type(ctype)
    tile = column_tile(h, ctype.item_size)
    if tile is None:
        raise ValueError(f"no column tile for {h} points")
    tiles = -(-m // tile.B)
    per = _images_per_workgroup(images, tiles + extra_tiles)
    groups = -(-images // per)
    nwg = (tiles + extra_tiles) * groups
    flag = lambda v: "true" if v else "false"  # noqa: E731
    pl = lambda rs: "vkx::PL<" + ", ".join(f"vkx::P<{r}, {ns}>" for r, ns in pass_list(rs)) + ">"  # noqa: E731
    lds = max(tile.lds_elems, 4 * h + h // tile.radices[0] + 1) if extra_tiles else tile.lds_elems
    lines = [
        "struct Cfg {",
        f"  using real = {real};",
        f"  static constexpr int N = {h}, TT = {tile.TT}, B = {tile.B}, BLOCK = {tile.TT * tile.B}, VMAX = {tile.vmax};",
        f"  static constexpr int PITCH = {tile.pitch}, LDS_ELEMS = {lds};",
        f"  static constexpr int M = {m}, SP = {m}, TILES = {tiles}, IMAGES = {images}, PER = {per}, "
        f"GROUPS = {groups};",
        f"  static constexpr bool KHALF = false, CONJ = {flag(conj)}, KEEP = {flag(keep)};",
        f"  static constexpr double SCALE = {1.0 / h!r};",
        f"  using fwd = {pl(list(tile.radices))};",
        f"  using inv = {pl(list(reversed(tile.radices)))};",
    ]
    if nwg % 8 == 0 and nwg >= 16:
        lines.append(f"  static constexpr bool XCDMAP = true; static constexpr vkx::u32 NWG = {nwg}u;")
    plan = KernelPlan(real=real, N=h, TT=tile.TT, B=tile.B, S=m, OUTER=images, radices=tile.radices, COLFAST=True,
                      WAVE_LOCAL=False, PAD_SHIFT=5, NP=0, LDS_ELEMS=lds, NWG=nwg, NWG_INNER=1)
    src = translation_unit("\n".join(lines + ["};"]), [], f"vkx::{body}<Cfg, {real}>(prm);", plan.BLOCK,
                           kernel_symbol(kind, plan, f"m{m}" + tag))
    src = src.replace('#include "vkx_fft.h"', '#include "vkx_half.h"')
    args = [Arg("output" if i == 0 else "input", "buffer", ctype, i) for i in range(slots_used)]
    kernel = CompiledKernel(src, plan, args, list(tile.radices), list(reversed(tile.radices)),
                            name=f"{kind}_{images}x{h}x{m}")
    kernel.groups = groups
    return kernel


@lru_cache(maxsize=None)
def make_half_conv(images: int, h: int, m: int, ctype, conj: bool = True, keep: bool = False) -> CompiledKernel:
    """Packed spectra [images][h][m] (slot 0, in place) down the columns: FFT, times packed K
    [h][m] (slot 1, conjugated if ``conj``), IFFT.  ``keep``: the transforms before the
    product go to slot 2, laid out like slot 0."""
    return _column_kernel("half_conv", "half_conv_body", h, m, images, ctype, 0, conj, 3 if keep else 2,
                          ("" if conj else "_nc") + ("_keep" if keep else ""), keep)


@lru_cache(maxsize=None)
def make_half_grad(images: int, h: int, m: int, ctype) -> CompiledKernel:
    """The adjoint over packed spectra [images][h][m]: g becomes dx (slot 0), the transforms
    X that the convolution kept (slot 1) and packed K (slot 2) are read, partial sums of dk go to slot 3, [kernel.groups][h][m]."""
    return _column_kernel("half_grad", "half_grad_body", h, m, images, ctype, 1, False, 4, "")


# ---- the whole convolution of an image in one workgroup -------------------------------
def _line_radices(n: int, lines: int) -> Optional[Tuple[Tuple[int, ...], int]]:
    """(radices, threads per line) of an n-point line within one wave: radices up to 16, the
    fewest passes, then the least idle work, then the threads that come nearest to a full
    workgroup over all ``lines`` (16 waves of 8 values 21 us, 8 waves of 16 values 23 us)."""
    for count in (1, 2, 3, 4):
        best = None
        for rads in groupings(n, count, 16):
            for tt in sorted({-(-n // (r * q)) for r in rads for q in (1, 2)}):
                values = max(slots(n, r, tt) for r in rads)
                if tt > 64 or values > 20:
                    continue
                waste = sum(slots(n, r, tt) * tt for r in rads) / (n * count) * 64 / (64 // tt * tt)
                key = (round(waste, 1), abs(math.log2(lines * tt / (64 * WHOLE_WAVES))), max(rads))
                if best is None or key < best[0]:
                    best = (key, rads, tt)
        if best is not None:
            return best[1:]
    return None


def _bank_conflicts(h: int, m: int, rows, cols, pitch: int) -> int:
    """Cycles of a wave's first exchange along a row and along a column: 64 lanes of 8 bytes
    over 32 pairs of banks, each direction's writes (a radix apart) and reads."""
    total = 0
    for (radices, tt), step, across in ((rows, 1, pitch), (cols, pitch, 1)):
        lanes = np.arange(64 // tt * tt)
        line, t = lanes // tt, lanes % tt
        for at in (t * radices[0], t):
            total += int(np.bincount((line * across + at * step) % 32, minlength=32).max())
    return total


@lru_cache(maxsize=None)
def whole_plan(h: int, m: int):
    """(rows, columns, LDS pitch) when an h x 2m image fits one workgroup, else None."""
    rows, cols = _line_radices(m, h), _line_radices(h, m)
    if rows is None or cols is None or h < 2 or m < 2:
        return None
    pitches = [p for p in range(m, m + 32) if 8 * (h * p + 2 * (h + m) + m) <= LDS_BYTES_MAX]
    if not pitches:
        return None
    # a second workgroup on the CU is worth more than the banks
    shared = [p for p in pitches if 8 * (h * p + 2 * (h + m) + m) <= LDS_SHARED]
    return rows, cols, min(shared or pitches, key=lambda p: (_bank_conflicts(h, m, rows, cols, p), p))


def _waves(h: int, m: int, row_threads: int, column_threads: int) -> int:
    """Waves of a workgroup that holds an h x 2m image: one for the lines of each."""
    return min(WHOLE_WAVES, max(-(-h // (64 // row_threads)), -(-m // (64 // column_threads))))


def whole_pays(images: int, h: int, m: int) -> bool:
    """Whether one workgroup per image beats three launches over all of them.  128^2: 256
    images 19.3 against 37.3 us, 96 17.9 / 19.5, 64 17.5 / 16.0 (the image alone takes 16.6, as
    long as one CU computes); 64^2: 1024 images 16.6 / 37, 4 images 8.2 / 10.  An image
    that leaves room for no second workgroup and few waves (160 x 200: 131 KB) is slower at
    any count.  From 513 images on a CU takes three and more of them in turn, while three launches
    gain on larger batches: 1024 images of 96^2 67 / 54 us, 800 of 96 x 120 67.5 / 56.5, but of
    128^2 68 / 79, of 64 x 128 28 / 47 (24 sizes, 12 counts of 96 to 1024)."""
    plan = whole_plan(h, m)
    if plan is None or 8 * h * plan[2] > WHOLE_LDS or (images < 96 and h * m > 4096):
        return False
    (rr, rtt), (cr, ctt), pitch = plan
    waves = _waves(h, m, rtt, ctt)
    side = min(LDS_BYTES_MAX // (8 * (h * pitch + 2 * (h + m) + m)), 32 // waves)
    if images <= 512 or h * m <= 2400 or side <= 1:
        return True
    # lines of a wave times the values of a thread, over the waves that a CU has at work on its
    # four SIMDs (5 and 6 waves of an image leave some of them idle)
    work = 2 * (-(-h // (64 // rtt)) * sum(slots(m, r, rtt) for r in rr) +
                -(-m // (64 // ctt)) * sum(slots(h, r, ctt) for r in cr))
    busy = min(32, waves * side) * waves / (4 * -(-waves // 4))
    points = images * h * 2 * m / 1e6
    return 4 + -(-images // 256) * 0.36 * work / busy < 1.05 * max(min(13 + 6.2 * points, 41), 5.3 * points)


class HalfWhole:
    """One launch: the convolution of each h x 2m image with a half spectrum (kstep elements
    from one image's to the next, 0: one for all), in place."""

    def __init__(self, images: int, h: int, m: int, kstep: int, normalize: bool):
        (rr, rtt), (cr, ctt), pitch = whole_plan(h, m)
        block = 64 * _waves(h, m, rtt, ctt)
        pl = lambda rs: "vkx::PL<" + ", ".join(f"vkx::P<{r}, {ns}>" for r, ns in pass_list(rs)) + ">"  # noqa: E731

        def line(name, n, radices, tt):
            vmax = max(slots(n, r, tt) for r in radices)
            return (f"  struct {name} {{ using real = float; static constexpr int N = {n}, TT = {tt}, VMAX = {vmax}; "
                    f"using fwd = {pl(list(radices))}; using inv = {pl(list(reversed(radices)))}; }};")
        cfg = "\n".join([
            "struct Cfg {",
            f"  static constexpr int N = {h}, M = {m}, RP = {pitch}, BLOCK = {block}, ROOTS = {math.lcm(2 * m, h)};",
            f"  static constexpr vkx::u64 IMG = {h * (2 * m + 2)}ull, KSTEP = {kstep}ull;",
            "  static constexpr bool KHALF = true, CONJ = true;",
            f"  static constexpr double SCALE = {1.0 / (2 * m * h) if normalize else 1.0!r};",
            line("RowCfg", m, rr, rtt), line("ColCfg", h, cr, ctt), "};"])
        plan = KernelPlan(real="float", N=m, TT=block, B=1, S=1, OUTER=images, radices=rr, COLFAST=False,
                          WAVE_LOCAL=False, PAD_SHIFT=5, NP=0, LDS_ELEMS=h * pitch, NWG=images, NWG_INNER=1)
        src = translation_unit(cfg, [], "vkx::half_whole_body<Cfg, float>(prm);", block,
                               kernel_symbol("half_whole", plan, f"h{h}" + ("" if kstep == 0 else "_k")))
        src = src.replace('#include "vkx_fft.h"', '#include "vkx_half.h"')
        args = [Arg("output" if i == 0 else "kernel", "buffer", dt.complex64, i) for i in range(2)]
        self.kernel = CompiledKernel(src, plan, args, None, None, name=f"half_whole_{images}x{h}x{2 * m}",
                                     roots_n=math.lcm(2 * m, h))

    def kernels(self):
        return [self.kernel]

    def values(self, buffer, kernel) -> list:
        return [buffer, kernel]


def clear() -> None:
    make_half_conv.cache_clear()
    make_half_grad.cache_clear()
    whole_plan.cache_clear()
