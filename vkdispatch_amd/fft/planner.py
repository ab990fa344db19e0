"""Plans for the gfx950 FFT kernels.

A plan fixes everything the kernel template needs at compile time: the radix
pass list (Stockham, each radix done in registers), the threads per transform
``TT``, the transforms per workgroup ``B``, the lane mapping (transform slot
fastest across lanes for strided axes, so every load is a contiguous run of
``B`` elements), the LDS layout and the launch grid.

Geometry follows the reference (vkdispatch/fft/config.py:217-233): a buffer of
shape ``shape`` transformed along ``axis`` is ``OUTER`` batches of ``N``
elements with stride ``S = prod(shape[axis+1:])`` (the ``S`` inner batches are
interleaved).  The plan choices themselves are this build's, made for wave64,
160 KB LDS and 256 CUs: the reference's register-budget search
(config.py:102-190) targets 32-wide subgroups and 32-64 KB of shared memory.
"""
from __future__ import annotations

import dataclasses
import math
import os
from functools import lru_cache
from typing import Iterator, List, Optional, Tuple

from .prime_utils import prime_factors

LDS_BYTES_MAX = 160 * 1024     # gfx950 LDS a workgroup may allocate
LDS_BYTES_TARGET = 64 * 1024   # keep >= 2 workgroups per CU when possible
MAX_THREADS = 1024
MAX_DIRECT_PRIME = 31          # larger primes go through Bluestein
WAVE = 64

# hand-picked power-of-two plans: N -> (radices, threads per transform)
_POW2 = {
    2: ([2], 1), 4: ([4], 1), 8: ([8], 1), 16: ([16], 1),
    32: ([8, 4], 4), 64: ([8, 8], 8), 128: ([16, 8], 8), 256: ([16, 16], 16),
    512: ([8, 8, 8], 64), 1024: ([16, 16, 4], 64), 2048: ([16, 16, 8], 128),
    4096: ([16, 16, 16], 256), 8192: ([16, 16, 16, 2], 512), 16384: ([16, 16, 16, 4], 1024),
}


def _wave_local_default() -> bool:
    return os.environ.get("VKX_WAVE_LOCAL", "1") != "0"


def groupings(n: int, count: int, most: int) -> Iterator[Tuple[int, ...]]:
    """The ways to write n as a product of ``count`` radices of at most ``most``, largest first."""
    def rec(rest: int, k: int, top: int):
        if k == 1:
            if 1 < rest <= top:
                yield (rest,)
            return
        for r in range(min(top, rest // 2 ** (k - 1)), 1, -1):
            if rest % r == 0:
                for tail in rec(rest // r, k - 1, r):
                    yield (r,) + tail
    yield from rec(n, count, most)


@lru_cache(maxsize=None)
def balanced_plan(N: int, elem: int) -> Optional[Tuple[Tuple[int, ...], int]]:
    """(radices, threads) of contiguous transforms whose length is no power of two: the
    least cost of the fewest passes, the idle slots and lanes in them, registers, barriers
    and short runs.  The weights are fitted to 1080 kernels of 61 lengths of 60 to 15000
    points, 50 MB in and out (MI355X): the picks are 1.3 % above the best of each length, the
    former rule (first-fit packing into radices up to 16, N / largest radix threads)
    26 %.  600 points 12.1 -> 10.3 us, 2160 17.0 -> 10.3, 480 15.3 -> 9.1; complex128 of
    600 points 12.7 -> 8.5, 2400 16.0 -> 10.2."""
    dbl = elem == 16
    most = 16 if dbl else 32     # values per thread: 64 registers
    if dbl and max(prime_factors(N)) > most:
        return None              # a butterfly of 17 or more complex128 needs more than that
    best = None
    for count in (2, 3, 4, 5):
        for rads in groupings(N, count, max(most, MAX_DIRECT_PRIME)):
            if any(r > most and len(prime_factors(r)) > 1 for r in rads):
                continue
            for order in {rads, rads[::-1]}:
                for tt in {-(-N // (r * q)) for r in rads for q in (1, 2, 3)}:
                    values = max(slots(N, r, tt) for r in order)
                    # 1024 threads leave 128 registers each, 512 leave 256
                    room = most if tt <= 512 else most // 2
                    if tt > MAX_THREADS or values > max(room, max(rads)) or values < 4:
                        continue
                    lanes = WAVE / (WAVE // tt * tt) if tt <= WAVE else -(-tt // WAVE) * WAVE / tt
                    work = sum(slots(N, r, tt) * tt for r in order) / N * lanes
                    cost = (0.1 * count + 0.223 * work + 0.464 * max(0, values - (12 if dbl else 20)) / most
                            + (0.05 if tt > WAVE else 0.0) + 0.1 * max(0.0, math.log2(128 / (tt * elem))))
                    key = (round(cost, 6), order, tt)
                    if best is None or key < best:
                        best = key
    return None if best is None else best[1:]


# values a thread may hold two sets of without spills, in workgroups of 513 to 1024, 257 to
# 512 and up to 256 threads (128, 256 and 512 registers; 2556 kernels of 142 lengths compiled)
_MOST_OF_TWO = ((13, 23, 32), (7, 14, 28))
UNEVEN_LDS = 44 * 1024  # up to here enough workgroups share a CU to even its four SIMDs out


@lru_cache(maxsize=None)
def column_radices(N: int, elem: int, B: int, live: int = 1) -> Optional[Tuple[Tuple[int, ...], int]]:
    """(radices, threads per transform) of strided transforms, B of them in a workgroup, that
    hold ``live`` sets of values at once: the
    cost of balanced_plan without what only concerns contiguous rows, the smaller radices
    first (512 = 16 32 points 8.9 us, 32 16 9.9; 320 columns, 50 MB in and out).  The idle
    lanes are those of the workgroup's last wave: 96 points 6 16 8.7 us, 8 12 7.5.  Two or
    three large workgroups on a CU want waves for all four SIMDs: 480 points of 24 threads
    (6 waves) 11.1 us, of 16 (4 waves) 9.2, convolved 18.2 and 15.5; complex128 432 points
    5 waves 10.8, 7 waves 8.2 us; at 280 and 320 points even waves lose 7 to 16 %."""
    dbl = elem == 16
    most = 16 if dbl else 32
    if dbl and max(prime_factors(N)) > most:
        return None
    best = None
    for count in (2, 3, 4, 5):
        for rads in groupings(N, count, max(most, MAX_DIRECT_PRIME)):
            if any(r > most and len(prime_factors(r)) > 1 for r in rads):
                continue
            for tt in {-(-N // (r * q)) for r in rads for q in (1, 2, 3)}:
                values = max(slots(N, r, tt) for r in rads)
                if tt * B > MAX_THREADS or values > max(most, max(rads)) or values < 4:
                    continue
                if tt * B > 512 and values > (12 if dbl else 20):  # at most 128 registers
                    continue
                if live > 1 and values > _MOST_OF_TWO[dbl][0 if tt * B > 512 else 1 if tt * B > 256 else 2]:
                    continue
                lanes = -(-tt * B // WAVE) * WAVE / (tt * B)
                work = sum(slots(N, r, tt) * tt for r in rads) / N * lanes
                waves = -(-tt * B // WAVE)
                uneven = -(-waves // 4) * 4 / waves - 1 if waves > 4 and B * N * elem > UNEVEN_LDS else 0.0
                cost = (0.1 * count + 0.223 * work + 0.464 * max(0, values - (12 if dbl else 20)) / most
                        + 0.38 * uneven)
                key = (round(cost, 6), rads[::-1], tt)
                if best is None or key < best:
                    best = key
    return None if best is None else best[1:]


def quick_radices(N: int, elem: int, passes: float) -> Iterator[Tuple[Tuple[int, ...], int]]:
    """(radices, threads per transform) by the time that one transform takes alone, ``passes``
    for each pass and 0.1 for each value of a thread: what a launch takes that does not fill the
    chip."""
    most = 16 if elem == 16 else 32
    found = []
    for count in (2, 3, 4):
        for rads in groupings(N, count, most):
            for tt in {-(-N // (r * q)) for r in rads for q in (1, 2, 3)}:
                held = [slots(N, r, tt) for r in rads]
                values = max(held)
                if tt > MAX_THREADS or values > most or values < max(4, max(rads)) or (tt > 512 and values > 16):
                    continue
                work = sum(held) * tt / (N * count)
                found.append((round(passes * count + 0.1 * values + 0.3 * (work - 1), 3), rads, tt))
    return ((rads, tt) for _, rads, tt in sorted(found))


FEW_POINTS = 1 << 19  # of a launch of rows; twice as many fill every SIMD


@lru_cache(maxsize=None)
def few_rows_plan(N: int, elem: int) -> Optional[Tuple[Tuple[int, ...], int]]:
    """(radices, threads) of launches of at most FEW_POINTS: three passes of up to 10 values
    rather than two of up to 32, one wave a workgroup.  25 lengths of 96 to 2000 points, real and
    complex, 2^14 to 2^19 points, against balanced_plan: 0.78 to 0.86 of the time (524 x 500 real
    points 7.1 -> 4.3 us, first-fit packing 5.1; 262 x 1000 complex 5.0 -> 3.8, 4.5); at 2^20 0.92,
    some lengths slower.  261 launches of random sizes: 68 took over 5 % more than with
    first-fit packing, 12 do."""
    return next(quick_radices(N, elem, 1.0), None)


def column_time(N: int, S: int, OUTER: int, elem: int, conv: bool, B: int, radices, tt: int) -> float:
    """Microseconds of a launch of strided transforms, B of them in a workgroup (fitted to 3264
    launches of 25 lengths of 96 to 2000, strides of 64 to 513, 0.02 to 6 M points: 15 % rms):
    rounds of workgroups times their own time, which is that of the values a thread handles
    and of the barriers of its size, and the bytes at the rate of a CU and of the chip, more
    of them where a tile is narrower than a cache line (much more where lines are not dealt to
    the XCDs in whole rows of tiles, as for aligned strides)."""
    held = [slots(N, r, tt) for r in radices]
    passes = 2 if conv else 1
    block = B * tt
    registers = max(held) * (13 if elem == 16 else 7.2 if conv else 6) + 16
    waves = max(1, min(8, int(512 // registers)), 4 if block > 768 else 3 if block > 512 else 2 if block > 256 else 1)
    lds = (N + (N - 1) // radices[0]) * B * elem
    side = max(1, min(LDS_BYTES_MAX // lds, 4 * waves // -(-block // WAVE), 2048 // block))
    tiles = OUTER * -(-S // B)
    each = -(-tiles // 256)
    width = B * elem / 8
    at4, at8 = (0.54, 0.23) if S * elem % 128 else (3.28, 1.07)
    more = 0.0 if width >= 16 else at8 * (16 - width) / 8 if width >= 8 else \
        at8 + (at4 - at8) * (8 - width) / 4 if width >= 4 else at4 * 4 / width
    moved = each * 2 * min(B, S) * N * elem / 117e3 + 2 * OUTER * N * S * elem / 11.65e6
    return 1.1 + -(-each // side) * (0.0615 * passes * sum(held) + 0.77 * block / 256) + moved * (1.0 + more)


@lru_cache(maxsize=None)
def column_plan(N: int, S: int, OUTER: int, elem: int, wide: int, conv: bool) -> Optional[Tuple[Tuple[int, ...], int, int]]:
    """(radices, threads per transform, transforms per workgroup) of a strided launch: the tile
    of ``wide`` transforms and its radices, or a narrower one, or fewer values a thread, where
    column_time makes that much shorter (at strides like those it was fitted to).  Few tiles, or a
    last round of large workgroups that is nearly empty, want more and smaller ones: 16 x 1000 x
    257 transformed 26.2 -> 18.7 us, convolved 40.5 -> 27.8 (first-fit packing 19.2, 27.8); 2 x 1000
    x 257 11.9 -> 6.4, 19.6 -> 9.0 (6.6, 9.1).  417 launches of random sizes: 64 took over 5 % more
    than with first-fit packing, 23 do (complex128 8 x 972 x 257 20.0 us, 15.0, among them)."""
    hit = column_radices(N, elem, wide)
    if hit is None or S < 32:
        return None if hit is None else (*hit, wide)
    (rads, tt), dbl = hit, elem == 16
    values, tiles = max(slots(N, r, tt) for r in rads), OUTER * -(-S // wide)
    # sure gains only: the formula does not know how a kernel was scheduled, and many tiles
    # leave less to gain (840 tiles of 252 points, predicted 0.85, took 1.11)
    bounded = fewer_waves(dbl, conv, S, wide, tt, values, tiles, N * wide * elem) is not None
    sure = 0.75 if bounded else 0.8 if tiles >= 512 else 0.9
    best = (sure * column_time(N, S, OUTER, elem, conv, wide, rads, tt), rads, tt, wide)
    quick = [(r[::-1], t) for (r, t), _ in zip(quick_radices(N, elem, 1.5), range(2))]
    for B in [wide] + [w // elem for w in ((64, 48) if dbl else (64, 48, 32)) if w // elem < wide]:
        hit = column_radices(N, elem, B)
        for rads, tt in quick + ([hit] if hit else []):
            values = max(slots(N, r, tt) for r in rads)
            if B * tt > MAX_THREADS or (B * tt > 512 and values > (9 if dbl else 16)):
                continue
            if (N + (N - 1) // rads[0]) * B * elem > LDS_BYTES_MAX:
                continue
            time = column_time(N, S, OUTER, elem, conv, B, rads, tt)
            if time < best[0]:
                best = (time, rads, tt, B)
    return best[1:]


def radix_plan(N: int) -> Tuple[List[int], int]:
    """(radices, threads-per-transform) for a length-N transform done in one workgroup."""
    if N < 1:
        raise ValueError("FFT length must be positive")
    if N == 1:
        return [1], 1
    if N in _POW2:
        r, t = _POW2[N]
        return list(r), t
    primes = prime_factors(N)
    if max(primes) > MAX_DIRECT_PRIME:
        raise ValueError(f"A prime factor of {N} is {max(primes)}, above the direct radix limit {MAX_DIRECT_PRIME}")
    if N <= 16:
        return [N], 1
    # first-fit-decreasing packing of the prime factors into radices <= 16
    radices: List[int] = []
    for p in sorted(primes, reverse=True):
        best = -1
        for i, r in enumerate(radices):
            if r * p <= 16 and (best < 0 or radices[i] > radices[best]):
                best = i
        if best >= 0:
            radices[best] *= p
        else:
            radices.append(p)
    radices.sort(reverse=True)
    tt = N // radices[0]
    return radices, max(1, tt)


def pass_list(radices: List[int]) -> List[Tuple[int, int]]:
    out, ns = [], 1
    for r in radices:
        out.append((r, ns))
        ns *= r
    return out


def slots(N: int, R: int, TT: int) -> int:
    W = N // R
    return -(-W // TT) * R


@dataclasses.dataclass(frozen=True)
class AxisGeometry:
    shape: Tuple[int, ...]
    axis: int
    N: int
    S: int       # stride between consecutive elements of one transform
    OUTER: int   # number of outer batches

    @staticmethod
    def of(shape, axis=None) -> "AxisGeometry":
        shape = tuple(int(s) for s in shape)
        if axis is None:
            axis = len(shape) - 1
        if axis < 0:
            axis += len(shape)
        if not 0 <= axis < len(shape):
            raise ValueError(f"axis {axis} out of range for shape {shape}")
        N = shape[axis]
        S = int(math.prod(shape[axis + 1:]))
        total = int(math.prod(shape))
        return AxisGeometry(shape, axis, N, S, total // (N * S))


@dataclasses.dataclass(frozen=True)
class KernelPlan:
    """Compile-time configuration of one FFT-family kernel (becomes ``struct Cfg``)."""
    real: str            # "float" | "double"
    N: int
    TT: int
    B: int
    S: int
    OUTER: int
    radices: Tuple[int, ...]
    COLFAST: bool
    WAVE_LOCAL: bool
    PAD_SHIFT: int
    NP: int
    LDS_ELEMS: int
    NWG: int
    NWG_INNER: int
    TWREG: bool = False  # twiddles in registers, loaded with the data (a tuned option)
    LPW: int = 0         # transforms of a wave whose last 64 - LPW TT lanes idle (0: none do)
    CPAD: bool = False   # COLFAST: LDS positions padded by B for every first radix of them

    @property
    def BLOCK(self) -> int:
        return self.B // self.LPW * WAVE if self.LPW else self.B * self.TT

    @property
    def fwd(self) -> List[Tuple[int, int]]:
        return pass_list(list(self.radices))

    @property
    def inv(self) -> List[Tuple[int, int]]:
        return pass_list(list(reversed(self.radices)))

    @property
    def VMAX(self) -> int:
        return max(slots(self.N, r, self.TT) for r in self.radices)

    @property
    def KSLOTS(self) -> int:
        return slots(self.N, self.radices[-1], self.TT)

    @property
    def lds_bytes(self) -> int:
        return self.LDS_ELEMS * (16 if self.real == "double" else 8)

    @property
    def grid(self) -> Tuple[int, int, int]:
        return (self.NWG, 1, 1)


_OVERRIDES: dict = {}
_TUNED: Optional[dict] = None


def plan_key(geom: AxisGeometry, real: str, kind: str) -> str:
    """Tuned plans depend on the transform length and stride, not on the batch count."""
    return f"{kind}|{geom.N}|{geom.S}|{real}"


def set_override(geom: AxisGeometry, real: str, kind: str, radices=None, tt=None, B=None, twreg=False) -> None:
    """Force a plan (used by the autotuner); ``radices=None`` removes the override.
    Kernel factories are cached: call ``vd.fft.cache_clear()`` after changing overrides."""
    key = plan_key(geom, real, kind)
    if radices is None:
        _OVERRIDES.pop(key, None)
    else:
        _OVERRIDES[key] = {"radices": list(radices), "tt": int(tt), "B": None if B is None else int(B),
                           "twreg": bool(twreg)}


def _tuned_table() -> dict:
    global _TUNED
    if _TUNED is None:
        import json
        path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuned_plans.json")
        try:
            with open(path) as f:
                _TUNED = json.load(f).get("plans", {})
        except (OSError, ValueError):
            _TUNED = {}
    return _TUNED


def lookup(geom: AxisGeometry, real: str, kind: str) -> Optional[dict]:
    key = plan_key(geom, real, kind)
    if key in _OVERRIDES:
        return _OVERRIDES[key]
    if os.environ.get("VKX_NO_TUNED") == "1":
        return None
    return _tuned_table().get(key)


def make_plan(geom: AxisGeometry, real: str = "float", batch_hint: Optional[int] = None,
              radices: Optional[List[int]] = None, tt: Optional[int] = None,
              need_lds: bool = False, kind: str = "fft", B_force: Optional[int] = None,
              transposed: bool = False, live: int = 1) -> KernelPlan:
    """Plan for ``geom``.  ``need_lds``: the kernel exchanges a full transform through
    LDS after its passes (real-FFT post-processing), so reserve B padded rows.
    ``kind`` selects the tuned-plan entry (autotuner results / overrides) if any.
    ``transposed``: a plan of the transposed-kernel layout, whose order follows from the
    threads and radices: these stay radix_plan's, so that stored kernels stay valid.
    ``live``: sets of values a thread of a strided kernel holds at once."""
    twreg = False
    if radices is None:
        hit = lookup(geom, real, kind)
        if hit is not None:
            radices, tt = hit["radices"], hit["tt"]
            B_force = hit.get("B") or B_force
            twreg = bool(hit.get("twreg", False))
    N, S, OUTER = geom.N, geom.S, geom.OUTER
    dbl = real == "double"
    elem = 16 if dbl else 8
    strided = S > 1
    if radices is None:
        if strided and N <= 32 and max(prime_factors(N) if N > 1 else [1]) <= MAX_DIRECT_PRIME:
            radices, tt = [N], 1
        else:
            radices, tt = radix_plan(N)
            if transposed:
                pass
            elif strided and tt <= MAX_THREADS:
                # whole 128-byte lines of neighbouring transforms before a second workgroup
                # on the CU: 1000 points 32.6 us at 5 of them, 11.9 at 16; complex128 of
                # 1024 16.9 at 4, 9.0 at 8.  Where that leaves a few large workgroups, whose
                # own time is what the launch takes, fewer of them: 320 columns of 1000 points
                # 10.4 us at 16, 8.2 at 8; 64 columns 10.1, 7.4 and at 4 6.7 (complex128: no gain)
                wide = min(S, 128 // elem)
                while wide > 1 and wide * N * elem > LDS_BYTES_MAX:
                    wide //= 2
                if not dbl and wide * N * elem > LDS_BYTES_TARGET:
                    most = 16 if S * OUTER > 512 else 8 if S * OUTER > 64 else 4
                    wide = min(wide, most)
                if live == 1:
                    hit = column_plan(N, S, OUTER, elem, wide, kind == "conv")
                    if hit is not None:
                        radices, tt, B_force = hit[0], hit[1], B_force or hit[2]
                else:
                    hit = column_radices(N, elem, wide, live)
                    while hit is None and wide > 4:
                        wide //= 2
                        hit = column_radices(N, elem, wide, live)
                    if hit is not None:
                        radices, tt = hit
                        B_force = B_force or wide
            elif N > 32 and N not in _POW2 and tt <= MAX_THREADS:
                few = OUTER * N <= FEW_POINTS and not dbl
                hit = few_rows_plan(N, elem) if few else balanced_plan(N, elem)
                if hit is not None:
                    radices, tt = hit
                    # two waves (one) when a wave holds whole transforms, else one transform a workgroup
                    B_force = B_force or ((1 if few else 2) * (WAVE // tt) if tt <= WAVE else 1)
    assert tt is not None
    radices = list(radices)
    if math.prod(radices) != N:
        raise ValueError(f"radices {radices} do not multiply to {N}")
    if tt > MAX_THREADS:
        raise ValueError(f"FFT of length {N} needs {tt} threads per transform (max {MAX_THREADS})")
    single_pass = len(radices) == 1
    pad_shift = 4 if elem == 16 else 5
    NP = N + (N >> pad_shift) + 1

    if strided:
        if tt == 1:
            B = min(S, 256)
        else:
            B = min(S, 16, max(1, MAX_THREADS // tt))
            while B > 1 and B * N * elem > LDS_BYTES_TARGET:
                B //= 2
        colfast = B > 1
    else:
        if tt == 1:
            B = 128 if N <= 8 else 64
        else:
            B = max(1, 256 // tt)
        B = max(1, min(B, OUTER))
        while B > 1 and (need_lds or not single_pass) and B * NP * elem > LDS_BYTES_TARGET:
            B //= 2
        colfast = False
    if batch_hint is not None:
        B = max(1, min(B, batch_hint))
    if B_force is not None:
        B = max(1, min(int(B_force), S if strided else OUTER, max(1, MAX_THREADS // tt)))
        colfast = strided and B > 1

    cpad = False
    if need_lds and not colfast:
        lds_elems = B * NP
    elif single_pass:
        lds_elems = 1
    elif colfast:
        lds_elems = N * B
        padded = (N + (N - 1) // radices[0]) * B
        # the padding against bank conflicts (512 points 10.3 -> 8.9 us) where it does not
        # take the place of a second workgroup (complex128 of 600 points 9.9 -> 11.7 us)
        if LDS_BYTES_MAX // (padded * elem) == LDS_BYTES_MAX // (lds_elems * elem) > 0:
            lds_elems, cpad = padded, True
    else:
        lds_elems = B * NP
    # A transform of at most 64 threads stays within a wave, whose exchanges need no barrier;
    # when the threads do not divide it, the wave's last lanes idle.
    wave_local = (not colfast) and tt <= WAVE and _wave_local_default()
    lpw = 0
    if transposed:
        wave_local = wave_local and WAVE % tt == 0
    elif wave_local and not strided and WAVE % tt:
        lpw = WAVE // tt
        B = max(lpw, min(-(-B // lpw), MAX_THREADS // WAVE) * lpw)
        while B > lpw and B * NP * elem > LDS_BYTES_TARGET:
            B -= lpw
        if lds_elems > 1:
            lds_elems = B * NP
    if lds_elems * elem > LDS_BYTES_MAX:
        raise ValueError(f"FFT of length {N} ({real}) needs {lds_elems * elem} bytes of LDS (max {LDS_BYTES_MAX})")

    if strided:
        nwg_inner = -(-S // B)
        nwg = OUTER * nwg_inner
    else:
        nwg_inner = 1
        nwg = -(-OUTER // B)
    if nwg >= 2 ** 31:
        raise ValueError("launch grid too large")
    return KernelPlan(real=real, N=N, TT=tt, B=B, S=S, OUTER=OUTER, radices=tuple(radices), COLFAST=colfast,
                      WAVE_LOCAL=wave_local, PAD_SHIFT=pad_shift, NP=NP, LDS_ELEMS=lds_elems, NWG=nwg,
                      NWG_INNER=nwg_inner, TWREG=twreg, LPW=lpw, CPAD=cpad)


def roomier_plans(geom: AxisGeometry, real: str, kind: str, need_lds: bool = False) -> Iterator[KernelPlan]:
    """Plans of fewer values a thread, for kernels that spill with the one they would have."""
    N, plan = geom.N, None
    radices, tt = ([N], 1) if geom.S > 1 and N <= 32 else radix_plan(N)
    for how in (dict(kind=kind, live=2), dict(radices=radices, tt=tt, transposed=True)):
        try:
            plan = make_plan(geom, real, need_lds=need_lds, **how)
        except ValueError:  # more threads or LDS than there are
            continue
        yield plan
    if plan is not None and plan.CPAD:  # the padded addresses take registers, too
        yield dataclasses.replace(plan, CPAD=False, LDS_ELEMS=plan.N * plan.B)


def overridden(geom: AxisGeometry, real: str, kind: str) -> bool:
    return plan_key(geom, real, kind) in _OVERRIDES


def wave_bounds(plan: KernelPlan, conv: bool) -> Optional[Tuple[int, int]]:
    """Least and most waves per SIMD to schedule a strided kernel for, or None: the
    compiler's own choice.  Where every tile is full (no guard keeps the loads together)
    and a thread holds many values, the compiler goes for four waves and up by putting
    each read of K and of a twiddle next to its use, up to 60 of them one after another,
    each waited for.  A launch that does not fill the chip has nothing to gain from more
    waves (1 x 640 x 320: convolved 13.7 -> 9.3 us, transformed 8.1 -> 6.3; 35 lengths of
    36 to 1024 convolved 14 % faster, the worst 2 % slower).  Others take three waves
    where they measured faster: convolutions with 24 values and up (26 x 500 x 320
    42.9 -> 30.7, 136 x 96 x 320 23.1 -> 15.8; with 20 and 21 values 300 to 400 points lose
    20 %, but 65 x 200 x 320, whose LDS allows six workgroups on a CU, 33.6 -> 19.3;
    workgroups of 8 waves have a second one on the CU only with four waves: 28.7 -> 31.3),
    complex128 transforms with 15 and 16 (40 x 160 x 320 14.4 -> 12.3, none slower than 2 %);
    complex64 transforms lose 4 %."""
    if not plan.COLFAST:
        return None
    return fewer_waves(plan.real == "double", conv, plan.S, plan.B, plan.TT, plan.VMAX, plan.NWG, plan.LDS_ELEMS * 8)


def fewer_waves(dbl: bool, conv: bool, S: int, B: int, tt: int, values: int, tiles: int,
                lds: int) -> Optional[Tuple[int, int]]:
    """wave_bounds of a strided plan."""
    block = B * tt
    if S % B or tt == 1 or block > 512 or values < (15 if dbl else 20):
        return None
    least = -(-block // (4 * WAVE))  # a workgroup's own
    if dbl:
        return None if conv else (least, 3)
    if tiles < 256:
        return least, 2
    if conv and block < 512 and (values >= 24 or (lds < 32 * 1024 and block > WAVE)):
        return least, 3
    return None


def whole_xcds(plan: KernelPlan) -> KernelPlan:
    """The plan with a grid of 8k workgroups (the last ones idle), as the XCD order needs."""
    return dataclasses.replace(plan, NWG=-(-plan.NWG // 8) * 8) if plan.NWG >= 16 else plan


def transposed_size(plan: KernelPlan) -> int:
    """Elements of the transposed-kernel layout consumed by a convolution with this plan."""
    return plan.NWG * plan.KSLOTS * plan.BLOCK
