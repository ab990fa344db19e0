"""Column kernels over packed half spectra (``csrc/device/vkx_half.h``): the middle of 2-D
real convolutions and of their adjoint, between the row kernels that write and read such
spectra (``make_real_rows_shader(..., packed=True)``)."""
from __future__ import annotations

from functools import lru_cache
from typing import Optional, Tuple

from .. import dtypes as dt
from .hooks import Arg
from .kernels import CompiledKernel, kernel_symbol, translation_unit
from .long import TilePlan, tile_radices
from .planner import LDS_BYTES_MAX, MAX_THREADS, KernelPlan, pass_list
from .precision import kernel_real_type

LDS_SHARED = 80 * 1024  # two workgroups on a CU
SLOTS = 512             # two workgroups on each CU


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


def _column_kernel(kind: str, body: str, h: int, m: int, pitch: int, images: int, ctype, extra_tiles: int, khalf: bool,
                   conj: bool, kstep: int, scale: float, slots_used: int, tag: str,
                   keep: bool = False) -> CompiledKernel:
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
        f"  static constexpr int M = {m}, SP = {pitch}, TILES = {tiles}, IMAGES = {images}, PER = {per}, "
        f"GROUPS = {groups};",
        f"  static constexpr vkx::u64 KSTEP = {kstep}ull;",
        f"  static constexpr bool KHALF = {flag(khalf)}, CONJ = {flag(conj)}, KEEP = {flag(keep)};",
        f"  static constexpr double SCALE = {scale!r};",
        f"  using fwd = {pl(list(tile.radices))};",
        f"  using inv = {pl(list(reversed(tile.radices)))};",
    ]
    if nwg % 8 == 0 and nwg >= 16:
        lines.append(f"  static constexpr bool XCDMAP = true; static constexpr vkx::u32 NWG = {nwg}u;")
    plan = KernelPlan(real=real, N=h, TT=tile.TT, B=tile.B, S=pitch, OUTER=images, radices=tile.radices, COLFAST=True,
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
def make_half_conv(images: int, h: int, m: int, pitch: int, ctype, khalf: bool, conj: bool = True, kstep: int = 0,
                   normalize: bool = True, keep: bool = False) -> CompiledKernel:
    """Spectra [images][h][pitch] (slot 0, m packed columns, in place) down the columns: FFT,
    times K (slot 1: a half spectrum [h][m + 1], or packed [h][m]; conjugated if ``conj``),
    IFFT.  ``keep``: the transforms before the product go to slot 2, laid out like slot 0."""
    return _column_kernel("half_conv", "half_conv_body", h, m, pitch, images, ctype, 0, khalf, conj, kstep,
                          1.0 / h if normalize else 1.0, 3 if keep else 2,
                          ("_k" if khalf else "") + ("" if conj else "_nc") + ("_keep" if keep else ""), keep)


@lru_cache(maxsize=None)
def make_half_grad(images: int, h: int, m: int, ctype) -> CompiledKernel:
    """The adjoint over packed spectra [images][h][m]: g becomes dx (slot 0), the transforms
    X that the convolution kept (slot 1) and packed K (slot 2) are read, partial sums of dk go to slot 3, [kernel.groups][h][m]."""
    return _column_kernel("half_grad", "half_grad_body", h, m, m, images, ctype, 1, False, False, 0, 1.0 / h, 4, "")


def clear() -> None:
    make_half_conv.cache_clear()
    make_half_grad.cache_clear()
