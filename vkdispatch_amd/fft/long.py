"""Uniform batches of transforms longer than one workgroup holds, in two launches.

A length L = n1 n2 runs as n1-point column transforms with the twiddles W_L^(k1 j2)
and n2-point row transforms (``csrc/device/vkx_long.h``), both compiled for the
length, so a transform crosses memory twice: 4 transforms of 2^20 points take 29 us
(15 + 13.5; a copy of the same bytes in two passes takes 16), where one workgroup
of the ragged executor took them through memory once per radix pass in 2.4 ms.
``split_length`` says how a length is cut; a length it cannot cut stays on the
ragged executor (``fft/ragged.py``).
"""
from __future__ import annotations

import dataclasses
import math
from functools import lru_cache
from typing import Dict, List, Optional, Tuple

from .. import dtypes as dt
from .. import runtime as rt
from ..buffer import Buffer
from .hooks import Arg
from .kernels import CompiledKernel, check_no_spill, kernel_symbol, translation_unit
from .planner import LDS_BYTES_MAX, MAX_THREADS, KernelPlan, groupings, pass_list, slots
from .prime_utils import prime_factors
from .scratch import SCRATCH_CAPTURES, SCRATCH_STREAMS, StreamScratch, launch_order  # noqa: F401

MAX_PRIME = 13        # larger prime factors go through Bluestein (fft/ragged.py)
MAX_RADIX = 32        # complex64 values a thread holds at most (64 registers)
TILE_MAX = 4096       # longest column or row: 4 of them (32-byte runs) still fit LDS
CHUNK_POINTS = 1 << 23  # points per pair of launches: 64 MiB of scratch, which stays in the 256 MB cache


@lru_cache(maxsize=None)
def tile_radices(n: int, most: int = MAX_RADIX) -> Optional[Tuple[Tuple[int, ...], int, float]]:
    """(radices, threads per transform, waste) of an n-point transform in registers: the
    fewest passes with at most ``most`` values per thread, then the least idle work.  ``waste`` is the butterflies' slots over
    their values (1: every thread has a full set in every pass)."""
    for count in (2, 3, 4):
        best = None
        for rads in groupings(n, count, MAX_RADIX):
            # three passes need no large radices, and these cost registers
            if count > 2 and max(rads) > 16 and n <= 16 ** count:
                continue
            for tt in sorted({n // (r * q) for r in rads for q in (1, 2, 3, 4) if n // (r * q) >= 4}):
                if tt > MAX_THREADS // 4 or max(slots(n, r, tt) for r in rads) > most:
                    continue
                waste = sum(slots(n, r, tt) * tt for r in rads) / (n * count)
                key = (round(waste, 2), max(rads), -tt)
                if best is None or key < best[0]:
                    best = (key, rads, tt, waste)
        if best is not None:
            return best[1:]
    return None


@dataclasses.dataclass(frozen=True)
class TilePlan:
    """One launch: transforms of length N, B of them per workgroup, TT threads each."""
    N: int
    radices: Tuple[int, ...]
    TT: int
    B: int
    turned: bool  # the tile is read the other way round in the last pass (column kernel)

    @property
    def pitch(self) -> int:
        return self.B + 1 if self.turned else self.B

    @property
    def lds_elems(self) -> int:
        return (self.N - 1) * self.pitch + (self.N - 1) // self.radices[0] * self.B + self.B

    @property
    def lds_bytes(self) -> int:
        return 8 * (self.lds_elems + (2 * self.B * self.radices[-1] if self.turned else 0))

    @property
    def vmax(self) -> int:
        return max(slots(self.N, r, self.TT) for r in self.radices)


def tile_plan(n: int, across: int, batch: int, turned: bool) -> Optional[TilePlan]:
    """Tile of an n-point launch over ``batch`` x ``across`` transforms.  16 transforms
    make 128-byte runs; 8 (64 bytes, joined in L2: neighbouring tiles run on one XCD) when
    16 do not fit LDS or leave CUs without a workgroup, 4 as the last resort."""
    hit = tile_radices(n)
    if hit is None:
        return None
    radices, tt, _ = hit
    fits = [t for t in (TilePlan(n, radices, tt, b, turned) for b in (16, 8, 4))
            if t.lds_bytes <= LDS_BYTES_MAX and t.TT * t.B <= MAX_THREADS]
    if not fits:
        return None
    for t in fits:
        if batch * -(-across // t.B) >= 256 or t.B == 8:
            return t
    return fits[-1]


# time of a launch over the same bytes, by length (4M points on MI355X): columns and rows of
# 512 points 13.6 / 12.7 us, 1024 14.5 / 13.5, 2048 17.2 / 16.4, 4096 about 25
def _launch_cost(n: int, waste: float, passes: int) -> float:
    base = 1.0 if n <= 512 else 1.07 if n <= 1024 else 1.28 if n <= 2048 else 1.9
    return base * (1.0 + 0.06 * max(0, passes - 2 - (n > 1024)) + 0.5 * (waste - 1.0))


@lru_cache(maxsize=None)
def split_length(n: int) -> Optional[Tuple[int, int]]:
    """(n1, n2) with n = n1 n2, both tiles of at most TILE_MAX points, or None."""
    if n < 4096 or max(prime_factors(n)) > MAX_PRIME:
        return None
    best = None
    for n1 in range(16, TILE_MAX + 1):
        if n % n1 or not 16 <= n // n1 <= TILE_MAX:
            continue
        n2 = n // n1
        cost = 0.0
        for m, turned in ((n1, True), (n2, False)):
            hit, tile = tile_radices(m), tile_plan(m, n // m, 1 << 20, turned)
            if hit is None or tile is None:
                break
            cost += _launch_cost(m, hit[2], len(hit[0])) * (1.0 if tile.B >= 8 or m > 2048 else 1.5)
        else:
            key = (round(cost, 3), abs(n1 - n2), n1)
            if best is None or key < best[0]:
                best = (key, (n1, n2))
    return best[1] if best else None


def _cfg(tile: TilePlan, n1: int, n2: int, b2: int, ys: int, nwg: int, tiles: int, inverse: bool,
         normalize: bool) -> str:
    flag = lambda v: "true" if v else "false"  # noqa: E731
    passes = ", ".join(f"vkx::P<{r}, {ns}>" for r, ns in pass_list(list(tile.radices)))
    lines = [
        "struct Cfg {",
        "  using real = float;",
        f"  static constexpr int N = {tile.N}, TT = {tile.TT}, B = {tile.B}, BLOCK = {tile.TT * tile.B}, "
        f"VMAX = {tile.vmax};",
        f"  static constexpr int PITCH = {tile.pitch}, LDS_ELEMS = {tile.lds_elems};",
        f"  static constexpr int N1 = {n1}, N2 = {n2}, B2 = {b2}, TILES = {tiles};",
        f"  static constexpr vkx::u64 YS = {ys}ull;",
        f"  static constexpr bool INV = {flag(inverse)}, NORMALIZE = {flag(normalize)};",
        f"  static constexpr double SCALE = {1.0 / (n1 * n2)!r};",
        f"  using fwd = vkx::PL<{passes}>;",
    ]
    # neighbouring tiles share cache lines when a run is shorter than a line or off it
    if nwg % 8 == 0 and nwg >= 16:
        lines.append(f"  static constexpr bool XCDMAP = true; static constexpr vkx::u32 NWG = {nwg}u;")
    return "\n".join(lines + ["};"])


def _kernel(tile: TilePlan, kind: str, body: str, cfg: str, nwg: int, batch: int, slots_used: int,
            tag: str) -> CompiledKernel:
    plan = KernelPlan(real="float", N=tile.N, TT=tile.TT, B=tile.B, S=1, OUTER=batch, radices=tile.radices,
                      COLFAST=True, WAVE_LOCAL=False, PAD_SHIFT=5, NP=0, LDS_ELEMS=tile.lds_elems, NWG=nwg,
                      NWG_INNER=1)
    src = translation_unit(cfg, [], body, plan.BLOCK, kernel_symbol(kind, plan, tag))
    src = src.replace('#include "vkx_fft.h"', '#include "vkx_long.h"')
    args = [Arg("output" if i == 0 else "input", "buffer", dt.complex64, i) for i in range(slots_used)]
    return CompiledKernel(src, plan, args, list(tile.radices), None, name=f"{kind}_{tile.N}x{batch}")


@lru_cache(maxsize=None)
def long_kernels(n: int, batch: int, inverse: bool, normalize: bool) -> Tuple[CompiledKernel, CompiledKernel]:
    """The column and row kernels of ``batch`` packed transforms of length n (no device needed)."""
    n1, n2 = split_length(n)
    cols = tile_plan(n1, n2, batch, True)
    rows = tile_plan(n2, n1, batch, False)
    ys = scratch_points(n, rows.B)
    tag = f"l{n}_" + ("inv" if inverse else "fwd")
    tiles = -(-n2 // cols.B)
    k_cols = _kernel(cols, "long_cols", f"vkx::long_cols_body<Cfg, vkx::PackedIn<1, {n}ull>>(prm);",
                     _cfg(cols, n1, n2, rows.B, ys, batch * tiles, tiles, inverse, False), batch * tiles, batch, 4,
                     tag)
    tiles = -(-n1 // rows.B)
    k_rows = _kernel(rows, "long_rows", f"vkx::long_rows_body<Cfg, vkx::PackedOut<0, {n}ull>>(prm);",
                     _cfg(rows, n1, n2, rows.B, ys, batch * tiles, tiles, inverse, inverse and normalize),
                     batch * tiles, batch, 2, tag)
    return k_cols, k_rows


def scratch_points(n: int, b2: int) -> int:
    """Elements between the launches per transform: whole tiles of b2 rows."""
    n1, n2 = split_length(n)
    return -(-n1 // b2) * b2 * n2


@lru_cache(maxsize=None)
def _twiddles(n: int, radix: int) -> Tuple[Buffer, Buffer]:
    """W_n^(j j2) as [j2][j], j < n1 / radix, and W_(radix n2)^(r j2) as [j2][r]: together
    W_n^(k1 j2) for k1 = j + r n1 / radix.  In FP64: the kernel rounds their product once."""
    n1, n2 = split_length(n)
    w = n1 // radix
    out = []
    for cols, step in ((w, 1), (radix, w)):
        b = Buffer((n2 * cols,), dt.complex128)
        rt.check(rt.lib().vkx_outer_roots(b.ptr, n2, cols, step, n, 1, rt.current_stream()), "vkx_outer_roots")
        out.append(b)
    rt.synchronize()
    return out[0], out[1]


class LongFFT(StreamScratch):
    """``count`` packed transforms of one length that split_length() cuts, in place in a
    complex64 buffer.  A batch of more than CHUNK_POINTS points runs in chunks of whole
    transforms, so that what lies between the launches stays in the cache."""

    def __init__(self, n: int, count: int, inverse: bool, normalize: bool):
        self.n, self.count = int(n), int(count)
        runs = -(-self.count // max(1, CHUNK_POINTS // self.n))
        each = -(-self.count // runs)
        self.chunks: List[Tuple[int, int]] = [(b, min(each, self.count - b)) for b in range(0, self.count, each)]
        self.kernels: Dict[int, Tuple[CompiledKernel, CompiledKernel]] = {
            c: long_kernels(self.n, c, bool(inverse), bool(normalize)) for _, c in self.chunks}
        for k in {k for pair in self.kernels.values() for k in pair}:
            check_no_spill(k)
        self.tables = _twiddles(self.n, self.kernels[each][0].plan.radices[-1])
        # whole row tiles of the largest chunk (the tile of a smaller one may be narrower)
        self._init_scratch(max(c * scratch_points(self.n, k[1].plan.B) for c, k in self.kernels.items()))

    def _new_scratch(self) -> Buffer:
        with rt.allocating_in_capture():  # launches may be recorded while a caller captures
            return Buffer((self._points,), dt.complex64)

    def _launches(self, buf, y) -> list:
        """(kernel, pointers) of every launch, through scratch ``y``."""
        if buf.size < self.n * self.count:
            raise ValueError(f"buffer of {buf.size} elements, the batch needs {self.n * self.count}")
        a, r = self.tables
        calls = []
        for first, c in self.chunks:
            cols, rows = self.kernels[c]
            x = int(buf.ptr) + 8 * self.n * first
            calls += [(cols, [y.ptr, x, a.ptr, r.ptr]), (rows, [x, y.ptr])]
        return calls

    def _load(self) -> None:
        for k in {k for pair in self.kernels.values() for k in pair}:
            k.handle()

    def bind(self, buf):
        """``launch(stream)`` for this buffer; it allocates nothing (safe under graph capture)
        and has scratch of its own: it may run on any stream, beside calls of this plan."""
        self._load()
        y = self._new_scratch()
        calls = self._launches(buf, y)
        keep = (buf, y, self)

        def launch(stream=None):
            _ = keep
            for k, ptrs in calls:
                k.launch_raw(ptrs, b"", stream)
        return launch

    def record(self, buf, graph) -> None:
        """Into a CommandGraph that is submitted later."""
        self._load()
        self._launches(buf, buf)  # refused now, not when it is submitted

        def launch(stream, y):
            for k, ptrs in self._launches(buf, y):
                k.launch_raw(ptrs, b"", stream)
        graph.record_with_scratch(launch, self._points)

    def __call__(self, buf) -> None:
        stream = rt.current_stream()
        with launch_order():
            y = self._scratch_for(stream)
            for k, ptrs in self._launches(buf, y):
                k.launch_raw(ptrs, b"", stream)


def clear() -> None:
    long_kernels.cache_clear()
    _twiddles.cache_clear()
