"""The workloads that speed is measured on: calls of the public entry points as a user's program makes them.

The ranges (``draw``): transforms of 64 to 2^20 points (powers of two, 7-smooth lengths, some primes), 2- and
3-D transforms and convolutions with sides of 32 to 1024, complex64 and complex128, 16-bit storage on the matrix
cores, differentiable convolutions and packed batches of mixed lengths.  In-place transforms run as a round trip
(forward, then inverse), so that a buffer can be transformed any number of times; convolution kernels have a
largest gain of 1 for the same reason.
"""
import functools
import math

import numpy as np
import torch

import vkdispatch_amd as vd
from vkdispatch_amd.fft import mixed, ragged
from vkdispatch_amd.fft.autograd import fft_convolve2d

_COMPLEX = {"c64": torch.complex64, "c128": torch.complex128}
_REAL = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # one call on a few short signals: the host path and the launches are all of it
        {"name": "c2c_8x256", "kind": "c2c", "batch": 8, "n": 256, "dtype": "c64"},
        # channels of a receiver, a power of two
        {"name": "c2c_1024x4096", "kind": "c2c", "batch": 1024, "n": 4096, "dtype": "c64"},
        # frames of a length that is chosen by its duration (30 ms at 50 kHz), not for the transform
        {"name": "c2c_2000x1500", "kind": "c2c", "batch": 2000, "n": 1500, "dtype": "c64"},
        # whole recordings, a million points each
        {"name": "c2c_4x1M", "kind": "c2c", "batch": 4, "n": 1 << 20, "dtype": "c64"},
        # images in double precision, sides that are no powers of two
        {"name": "fft2_c128_8x600x800", "kind": "fftn", "batch": 8, "h": 600, "w": 800, "d": 0, "dtype": "c128"},
        # the volume of a spectral solver: there and back
        {"name": "fft3_256", "kind": "fftn", "batch": 0, "h": 256, "w": 256, "d": 256, "dtype": "c64"},
        # the same volume held in 16 bits, transformed on the matrix cores
        {"name": "mixed3d_bf16_256", "kind": "mixed", "storage": "bf16", "inverse": False},
        # the headline workload: one blur kernel over a batch of square images
        {"name": "conv_64x512x512", "kind": "conv", "batch": 64, "h": 512, "w": 512},
        # video frames
        {"name": "conv_24x480x640", "kind": "conv", "batch": 24, "h": 480, "w": 640},
        # patches of a larger picture
        {"name": "conv_256x128x128", "kind": "conv", "batch": 256, "h": 128, "w": 128},
        # one training step of a learnable kernel as large as the images: output, and both gradients
        {"name": "grad_32x1024x1024", "kind": "grad", "batch": 32, "h": 1024, "w": 1024, "dtype": "f32"},
        # a packed batch of mixed lengths, primes among them, replayed as a graph
        {"name": "ragged_4096", "kind": "ragged", "count": 4096, "mix": 0},
    ]


# ---- drawn cases --------------------------------------------------------------------
def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _prime(n):
    return n > 1 and all(n % d for d in range(2, int(n ** 0.5) + 1))


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi, primes=False, even=False):
    """A length of [lo, hi]: a power of two, a 7-smooth number or (primes) a prime."""
    u = rng.random()
    if u < 0.4:
        return 2 ** rng.randint(math.ceil(math.log2(lo)), math.floor(math.log2(hi)))
    if primes and u > 0.9:
        n = _log_uniform(rng, lo, min(hi, 60000))
        while not _prime(n):
            n += 1
        return n
    n = _log_uniform(rng, lo, hi)
    while not (_smooth(n) and (n % 2 == 0 or not even)):
        n -= 1
    return max(n, lo)


def _batch(rng, size, lo, hi, most=4096):
    """How many signals of ``size`` points make between lo and hi points."""
    return max(1, min(most, _log_uniform(rng, max(lo, size), max(hi, size)) // size))


def draw(rng):
    kind = rng.choices(["c2c", "fft2", "fft3", "conv", "grad", "mixed", "ragged"], [5, 2, 1.5, 5, 1.5, 0.5, 1])[0]
    if kind == "c2c":
        if rng.random() < 0.2:
            n = _length(rng, 64, 4096)
            return {"kind": "c2c", "batch": _batch(rng, n, 1 << 11, 1 << 21), "n": n, "dtype": "c128"}
        n = _length(rng, 64, 1 << 20, primes=True)
        return {"kind": "c2c", "batch": _batch(rng, n, 1 << 11, 1 << 22), "n": n, "dtype": "c64"}
    if kind == "fft2":
        h, w = _length(rng, 32, 1024), _length(rng, 32, 1024)
        dtype = rng.choice(["c64", "c64", "c128"])
        return {"kind": "fftn", "batch": _batch(rng, h * w, 1 << 14, 1 << 22), "h": h, "w": w, "d": 0, "dtype": dtype}
    if kind == "fft3":
        return {"kind": "fftn", "batch": 0, "h": _length(rng, 32, 256), "w": _length(rng, 32, 256),
                "d": _length(rng, 32, 256), "dtype": "c64"}
    if kind == "conv":
        h = _length(rng, 32, 1024)
        w = h if rng.random() < 0.5 else _length(rng, 32, 1024)
        return {"kind": "conv", "batch": _batch(rng, h * w, 1 << 14, 1 << 24, 1024), "h": h, "w": w}
    if kind == "grad":
        h, w = _length(rng, 64, 1024), _length(rng, 64, 1024, even=True)
        dtype = rng.choice(["f32", "f32", "f32", "f64"])
        return {"kind": "grad", "batch": _batch(rng, h * w, 1 << 16, 1 << 23, 64), "h": h, "w": w, "dtype": dtype}
    if kind == "mixed":
        storage, inverse = rng.choice([("bf16", True), ("fp16", False), ("fp16", True)])
        return {"kind": "mixed", "storage": storage, "inverse": inverse}
    return {"kind": "ragged", "count": _log_uniform(rng, 128, 2048), "mix": rng.randint(1, 1 << 20)}


# ---- inputs (from the seed alone) ---------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _shape(case):
    if case["kind"] == "c2c":
        return (case["batch"], case["n"])
    if case["d"]:
        return (case["h"], case["w"], case["d"])
    return (case["batch"], case["h"], case["w"])


def _normal(case, seed, shape=None):
    return torch.randn(shape or _shape(case), dtype=_COMPLEX[case.get("dtype", "c64")], device="cuda",
                       generator=_generator(seed))


def _images(case, seed):
    """Images U(-1, 1) and the half spectrum of a blur kernel with noise, its largest gain 1."""
    g, h, w = _generator(seed), case["h"], case["w"]
    x = torch.rand((case["batch"], h, w), device="cuda", generator=g) * 2 - 1
    y0, x0 = torch.arange(h, device="cuda").double(), torch.arange(w, device="cuda").double()
    dy, dx = torch.minimum(y0, h - y0)[:, None], torch.minimum(x0, w - x0)[None, :]
    k = torch.exp(-(dy ** 2 + dx ** 2) / (2 * 4.0 ** 2))
    k = k + 0.01 * torch.randn((h, w), device="cuda", generator=g).double()
    kf = torch.fft.rfft2(k)
    return x, (kf / kf.abs().max()).to(torch.complex64).contiguous()


def _grad_inputs(case, seed):
    g, shape, dtype = _generator(seed), (case["batch"], case["h"], case["w"]), _REAL[case["dtype"]]
    x = torch.randn(shape, dtype=dtype, device="cuda", generator=g)
    k = 0.01 * torch.randn(shape[1:], dtype=dtype, device="cuda", generator=g)
    return x, k, torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _volume(case, seed):
    """A 256^3 volume as the (real, imaginary) pairs of its storage."""
    dtype = torch.bfloat16 if case["storage"] == "bf16" else torch.float16
    return torch.randn((256, 256, 256, 2), device="cuda", generator=_generator(seed)).to(dtype)


@functools.lru_cache(maxsize=4)
def _sizes(count, mix):
    return tuple(ragged.mixed_sizes(count, seed=mix))


@functools.lru_cache(maxsize=1)
def _ragged_plan(count, mix):
    """One plan for a list of lengths, kept over its inputs."""
    return ragged.RaggedFFT(_sizes(count, mix))


# ---- the cases ----------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("c2c", "fftn"):
        x = _normal(case, seed)
        return {"case": case, "x": x, "buf": vd.from_cuda_array(x)}
    if kind == "mixed":
        pairs = _volume(case, seed)
        vt = vd.complex_bf16 if case["storage"] == "bf16" else vd.complex32
        inp = vd.Buffer((256, 256, 256), vt)
        inp.to_torch().copy_(pairs)
        out = torch.empty((256, 256, 256), dtype=torch.complex64, device="cuda")
        return {"case": case, "inp": inp, "out": out, "buf": vd.from_cuda_array(out)}
    if kind == "conv":
        x, kf = _images(case, seed)
        rows = torch.zeros(x.shape[:-1] + (2 * (case["w"] // 2 + 1),), device="cuda")
        rows[..., :case["w"]] = x
        return {"case": case, "y": rows[..., :case["w"]],
                "buf": vd.rfftbuffer_from_cuda_array(rows, tuple(x.shape)),
                "kernel": vd.rfftbuffer_from_cuda_array(kf, (case["h"], case["w"]))}
    if kind == "grad":
        x, k, g = _grad_inputs(case, seed)
        return {"case": case, "x": x.requires_grad_(), "k": k.requires_grad_(), "g": g}
    plan = _ragged_plan(case["count"], case["mix"])
    x = _normal(case, seed, (plan.total,))
    y = torch.empty_like(x)
    out, inp = vd.from_cuda_array(y), vd.from_cuda_array(x)
    graph = vd.CommandGraph()
    graph.record_callable(plan.bind(out, inp))
    graph.capture()
    return {"case": case, "y": y, "graph": graph, "bufs": (out, inp)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "c2c":
        vd.fft.fft(state["buf"])
        vd.fft.ifft(state["buf"])
        return state["x"]
    if kind == "fftn":
        forward, inverse = (vd.fft.fft3, vd.fft.ifft3) if case["d"] else (vd.fft.fft2, vd.fft.ifft2)
        forward(state["buf"])
        inverse(state["buf"])
        return state["x"]
    if kind == "mixed":
        mixed.fft3_mixed(state["buf"], state["inp"], inverse=case["inverse"])
        return state["out"]
    if kind == "conv":
        vd.fft.convolve2DR(state["buf"], state["kernel"], kernel_inner_only=True)
        return state["y"]
    if kind == "grad":
        y = fft_convolve2d(state["x"], state["k"])
        dx, dk = torch.autograd.grad(y, (state["x"], state["k"]), state["g"])
        return {"y": y, "dx": dx, "dk": dk}
    state["graph"].submit()
    return state["y"]


# ---- what a pass cannot do without: inputs read once, outputs written once ------------
def work(case):
    kind = case["kind"]
    if kind in ("c2c", "fftn"):  # forward and inverse
        shape = _shape(case)
        points = math.prod(shape)
        along = shape[1:] if kind == "c2c" or not case["d"] else shape
        item = 16 if case["dtype"] == "c128" else 8
        return {"bytes": 4 * item * points, "flops": 2 * 5 * points * sum(math.log2(n) for n in along)}
    if kind == "mixed":
        points = 256 ** 3
        return {"bytes": (4 + 8) * points, "flops": 5 * points * 24}
    if kind == "conv":
        points, plane = case["batch"] * case["h"] * case["w"], case["h"] * (case["w"] // 2 + 1)
        return {"bytes": 8 * points + 8 * plane, "flops": points * (5 * math.log2(case["h"] * case["w"]) + 3)}
    if kind == "grad":
        points, plane = case["batch"] * case["h"] * case["w"], case["h"] * case["w"]
        item = 8 if case["dtype"] == "f64" else 4
        # x, k in, y out; then g, x in, dx, dk out
        return {"bytes": item * (5 * points + 2 * plane),
                "flops": points * (12.5 * math.log2(case["h"] * case["w"]) + 9)}
    sizes = np.array(_sizes(case["count"], case["mix"]), dtype=np.float64)
    return {"bytes": float(16 * sizes.sum()), "flops": float((5 * sizes * np.log2(sizes)).sum())}


# ---- the same in 64 bits ------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind in ("c2c", "fftn"):  # the round trip ends where it began
        return _normal(case, seed).to(torch.complex128)
    if kind == "mixed":
        z = torch.view_as_complex(_volume(case, seed).double())
        return torch.fft.ifftn(z) if case["inverse"] else torch.fft.fftn(z)
    if kind == "conv":
        x, kf = _images(case, seed)
        size = (case["h"], case["w"])
        return torch.cat([torch.fft.irfft2(torch.fft.rfft2(p.double()) * kf.to(torch.complex128).conj(), s=size)
                          for p in x.split(16)])
    if kind == "grad":
        x, k, g = (t.double() for t in _grad_inputs(case, seed))
        size = (case["h"], case["w"])
        xf, kf, gf = torch.fft.rfft2(x), torch.fft.rfft2(k), torch.fft.rfft2(g)
        return {"y": torch.fft.irfft2(xf * kf.conj(), s=size), "dx": torch.fft.irfft2(gf * kf, s=size),
                "dk": torch.fft.irfft2((xf * gf.conj()).sum(0), s=size)}
    sizes = _sizes(case["count"], case["mix"])
    x = _normal(case, seed, (sum(sizes),)).cpu().numpy().astype(np.complex128)
    ends = np.cumsum(sizes)
    return np.concatenate([np.fft.fft(p) for p in np.split(x, ends[:-1])])
