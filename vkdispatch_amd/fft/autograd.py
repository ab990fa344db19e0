"""Differentiable FFT-convolution with a hand-written adjoint.

``fft_convolve2d(x, k)`` computes, per image, the vd.fft.convolve2DR result

    y = irfft2(rfft2(x) * conj(rfft2(k)))     i.e.  y[n] = sum_m x[n + m] k[m]

(circular cross-correlation, the reference's default convolution kernel map,
vkdispatch/fft/shader_factories.py:136-145) for real ``x`` of shape
(..., H, W) and a real kernel ``k`` of shape (H, W) broadcast over the batch.

Backward (adjoint of a cross-correlation):
    dx = irfft2(rfft2(g) * K)                              (convolution with k)
    dk = sum_b irfft2(rfft2(x_b) * conj(rfft2(g_b)))       (correlation of x with g)
with K = rfft2(k) and g = dL/dy.

Everything runs on the gfx950 kernels of this package, on PyTorch's current
stream, with PyTorch providing only the tensors (storage) and autograd:
  forward  : rows r2c (out of place) -> column FFT * conj(K) -> column IFFT (one
             fused kernel) -> rows c2r (out of place)
  backward : rows r2c of g -> one column kernel with its FFT, IFFT of
             G * K and IFFTs of partial sums of X * conj(G) over the batch (X kept by
             the forward column kernel) -> rows c2r of dx, and of dk from the sum of
             the partial sums (_HalfPlans); or with a column kernel for each of these
             (_Plans, for heights without a column tile).
"""
from __future__ import annotations

import ctypes
from functools import lru_cache

from .. import codegen as vc
from .. import dtypes as dt
from .. import runtime as rt
from ..buffer import Buffer
from ..shader_map import map as vd_map
from . import functions as F
from . import half2d
from .kernels import SpillError, check_no_spill
from .shader_factories import make_convolution_shader, make_fft_shader, make_real_rows_shader, register_plan_cache


def _torch():
    import torch
    return torch


def _ctype(real_dtype):
    torch = _torch()
    if real_dtype == torch.float32:
        return dt.complex64, torch.complex64
    if real_dtype == torch.float64:
        return dt.complex128, torch.complex128
    raise TypeError(f"fft_convolve2d supports float32 and float64 tensors, got {real_dtype}")


def _wrap(t, var_type, shape=None) -> Buffer:
    """Zero-copy Buffer over a contiguous CUDA tensor."""
    if not t.is_cuda or not t.is_contiguous():
        raise ValueError("fft_convolve2d needs contiguous device tensors")
    return Buffer(tuple(shape if shape is not None else t.shape), var_type, external=(t.data_ptr(), t, True))


@lru_cache(maxsize=None)
def _mult_kernel_map(img_elems: int, ctype):
    """Input map: load the spectrum element and multiply by K (not conjugated), K
    broadcast over the batch (index = io_index mod H*(W/2+1))."""
    from .hooks import read_op

    def mult_k(spec, kern):
        op = read_op()
        op.read_from_buffer(spec)
        kv = vc.to_dtype(op.register.var_type, kern[op.io_index % img_elems])
        op.register[:] = vc.mult_complex(op.register, kv)
    return vd_map(mult_k, input_types=[vc.Buffer[ctype], vc.Buffer[ctype]])


class _Plans:
    def __init__(self, B, H, W, ctype):
        self.B, self.H, self.W = B, H, W
        Wh = W // 2 + 1
        self.Wh = Wh
        self.ctype = ctype
        c = ctype
        self.rows_fwd = make_real_rows_shader((B, H, W), False, True, c, c, True, W, Wh)
        self.rows_inv = make_real_rows_shader((B, H, W), True, True, c, c, True, W, Wh)
        self.rows_fwd1 = make_real_rows_shader((1, H, W), False, True, c, c, True, W, Wh)
        self.rows_inv1 = make_real_rows_shader((1, H, W), True, True, c, c, True, W, Wh)
        self.col_fft1 = make_fft_shader((1, H, Wh), 1, input_type=c, output_type=c, compute_type=c)
        self.col_fft = make_fft_shader((B, H, Wh), 1, input_type=c, output_type=c, compute_type=c)
        self.conv_bcast = make_convolution_shader((B, H, Wh), None, 1, 1, kernel_inner_only=True, input_type=c,
                                                  output_type=c, kernel_type=c, compute_type=c)
        self.conv_full = make_convolution_shader((B, H, Wh), None, 1, 1, input_type=c, output_type=c,
                                                 kernel_type=c, compute_type=c)
        self.kmap = _mult_kernel_map(H * Wh, c)

    def kernels(self):
        dx = make_fft_shader((self.B, self.H, self.Wh), 1, inverse=True, input_map=self.kmap,
                             output_type=self.ctype, compute_type=self.ctype)
        return [self.rows_fwd, self.rows_inv, self.rows_fwd1, self.rows_inv1, self.col_fft1, self.col_fft,
                self.conv_bcast, self.conv_full, dx]

    def forward(self, x, ws, K, keep):
        """Columns of ws; returns what the gradient of k needs of x."""
        self.conv_bcast.launch([ws, K])
        return x if keep else None

    def backward(self, x, K, g, Gb, need_dx, need_dk):
        torch = _torch()
        real_t = self.ctype.child_type
        self.col_fft.launch([Gb])                           # rfft2(g)
        dx = dk = None
        if need_dk:
            wb = _wrap(_spectra(self, self.B, x.device), self.ctype)
            self.rows_fwd.launch([wb, _wrap(x, real_t)])
            self.conv_full.launch([wb, Gb])                 # col-IFFT(rfft2(x_b) * conj(G_b))
            dk = _summed_rows(self, wb, self.B, g)
        if need_dx:
            # column IFFT of G * K (K applied by the input map), in place, then rows c2r
            F.fft(Gb, Gb, K, axis=1, inverse=True, input_map=self.kmap)
            dx = torch.empty_like(g)
            self.rows_inv.launch([_wrap(dx, real_t), Gb])
        return dx, dk


class _HalfPlans:
    """The same convolution on packed half spectra (fft/half2d.py): W / 2 columns in whole
    tiles, aligned, and one column launch for the whole adjoint.  32 x 1024^2 in a training
    step (kernel trace): the forward column launch 74 us (96 with W / 2 + 1 columns; 111 when
    it also stores X), the adjoint's 147 us for 295 us of separate transforms, products and
    batch sum and 58 us of rows of x; the step 682 -> 550 us."""

    def __init__(self, B, H, W, ctype):
        self.B, self.H, self.W = B, H, W
        self.Wh = M = W // 2  # columns of a spectrum
        self.ctype = c = ctype
        self.rows_fwd = make_real_rows_shader((B, H, W), False, True, c, c, True, W, M, True)
        self.rows_inv = make_real_rows_shader((B, H, W), True, True, c, c, True, W, M, True)
        self.rows_fwd1 = make_real_rows_shader((1, H, W), False, True, c, c, True, W, M, True)
        self.col_fft1 = make_fft_shader((1, H, M), 1, input_type=c, output_type=c, compute_type=c)
        self.conv = half2d.make_half_conv(B, H, M, c)
        self.conv_keep = half2d.make_half_conv(B, H, M, c, keep=True)
        self.conv_dx = half2d.make_half_conv(B, H, M, c, conj=False)
        self.grad = half2d.make_half_grad(B, H, M, c)
        self.rows_inv1 = make_real_rows_shader((1, H, W), True, True, c, c, True, W, M, True)
        self._fits = {}

    def fits(self, kernel) -> bool:
        """Whether a launch that does part of another's work compiles without spills, found out
        when it is first wanted (plans_for has compiled the others)."""
        if kernel not in self._fits:
            try:
                check_no_spill(kernel)
                self._fits[kernel] = True
            except SpillError:
                self._fits[kernel] = False
        return self._fits[kernel]

    def kernels(self):
        return [self.rows_fwd, self.rows_inv, self.rows_fwd1, self.col_fft1, self.conv, self.conv_keep,
                self.conv_dx, self.grad, self.rows_inv1]

    def forward(self, x, ws, K, keep):
        """Columns of ws; returns what the gradient of k needs of x: its transform, which the
        column kernel has at hand.  It takes the place of x between the passes."""
        if not keep and self.fits(self.conv):
            self.conv.launch([ws, K])
            return None
        X = _spectra(self, self.B, x.device)
        self.conv_keep.launch([ws, K, _wrap(X, self.ctype)])
        return X if keep else None

    def backward(self, X, K, g, Gb, need_dx, need_dk):
        torch = _torch()
        dx = dk = None
        if need_dk or not self.fits(self.conv_dx):
            partial = _wrap(_spectra(self, self.grad.groups, g.device), self.ctype)
            # where dk is not wanted its sum is of anything: of G
            self.grad.launch([Gb, _wrap(X, self.ctype) if need_dk else Gb, K, partial])
        else:
            self.conv_dx.launch([Gb, K])
        if need_dx:
            dx = torch.empty_like(g)
            self.rows_inv.launch([_wrap(dx, self.ctype.child_type), Gb])
        if need_dk:
            dk = _summed_rows(self, partial, self.grad.groups, g)
        return dx, dk


def _summed_rows(plans, spectra, count, g):
    """dk from ``count`` column-transformed spectra: their sum (in a fixed order), then rows c2r."""
    torch = _torch()
    dbl = 1 if plans.ctype is dt.complex128 else 0
    P = _wrap(_spectra(plans, 1, g.device), plans.ctype)
    rt.check(rt.lib().vkx_batch_sum(P.ptr, spectra.ptr, count, 2 * plans.H * plans.Wh, dbl, rt.current_stream()),
             "vkx_batch_sum")
    dk = torch.empty((plans.H, plans.W), dtype=g.dtype, device=g.device)
    plans.rows_inv1.launch([_wrap(dk, plans.ctype.child_type), P])
    return dk


@lru_cache(maxsize=64)
def plans_for(B, H, W, ctype):
    if W % 2:
        raise ValueError("fft_convolve2d needs an even last dimension")
    if half2d.column_tile(H, ctype.item_size) is not None:
        try:
            plans = _HalfPlans(B, H, W, ctype)
            for k in (plans.conv_keep, plans.grad):
                check_no_spill(k)
            return plans
        except (SpillError, ValueError):  # a length whose kernel does not fit the registers or the LDS
            pass
    return _Plans(B, H, W, ctype)


register_plan_cache(plans_for.cache_clear)
register_plan_cache(half2d.clear)


def _spectra(plans, images, device):
    """Tensor of the spectra of ``images`` images in the plan's layout."""
    torch = _torch()
    tct = torch.complex128 if plans.ctype is dt.complex128 else torch.complex64
    return torch.empty((images, plans.H, plans.Wh), dtype=tct, device=device)


def kernel_spectrum(k, plans):
    """K = rfft2(k) for a (H, W) real tensor, as a (H, plans.Wh) complex tensor in the
    plan's layout."""
    K = _spectra(plans, 1, k.device)[0]
    Kb = _wrap(K, plans.ctype)
    plans.rows_fwd1.launch([Kb, _wrap(k, plans.ctype.child_type)])
    plans.col_fft1.launch([Kb])
    return K


def _forward(x, k, plans, keep=False):
    """y, K and, with ``keep``, what the gradient of k needs of x."""
    torch = _torch()
    real_t = plans.ctype.child_type
    K = kernel_spectrum(k, plans)
    ws = _wrap(_spectra(plans, plans.B, x.device), plans.ctype)
    plans.rows_fwd.launch([ws, _wrap(x, real_t)])
    kept = plans.forward(x, ws, _wrap(K, plans.ctype), keep)
    y = torch.empty_like(x)
    plans.rows_inv.launch([_wrap(y, real_t), ws])
    return y, K, kept


def _backward(kept, K, g, plans, need_dx: bool, need_dk: bool):
    if not (need_dx or need_dk):
        return None, None
    Gb = _wrap(_spectra(plans, plans.B, g.device), plans.ctype)
    plans.rows_fwd.launch([Gb, _wrap(g, plans.ctype.child_type)])
    return plans.backward(kept, _wrap(K, plans.ctype), g, Gb, need_dx, need_dk)


def _run(fn, *args):
    torch = _torch()
    with rt.stream_scope(torch.cuda.current_stream()):
        return fn(*args)


def _autograd_function():
    torch = _torch()

    class FFTConvolve2DFunction(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, k, recorded):
            shape = x.shape
            H, W = shape[-2], shape[-1]
            if tuple(k.shape) != (H, W):
                raise ValueError(f"kernel shape {tuple(k.shape)} must equal the image shape {(H, W)}")
            if x.dtype != k.dtype:
                raise TypeError("x and k must have the same dtype")
            ctype, _ = _ctype(x.dtype)
            x3 = x.contiguous().reshape(-1, H, W)
            kc = k.contiguous()
            plans = plans_for(x3.shape[0], H, W, ctype)
            y, K, kept = _run(_forward, x3, kc, plans,
                              recorded and ctx.needs_input_grad[1])
            ctx.save_for_backward(kept, K)
            ctx.plans = plans
            ctx.in_shape = shape
            return y.reshape(shape)

        @staticmethod
        def backward(ctx, gy):
            kept, K = ctx.saved_tensors
            plans = ctx.plans
            g3 = gy.contiguous().reshape(plans.B, plans.H, plans.W)
            dx, dk = _run(_backward, kept, K, g3, plans, ctx.needs_input_grad[0], ctx.needs_input_grad[1])
            if dx is not None:
                dx = dx.reshape(ctx.in_shape)
            return dx, dk, None

    return FFTConvolve2DFunction


_FN = None


def fft_convolve2d(x, k):
    """Differentiable ``irfft2(rfft2(x) * conj(rfft2(k)))`` over the last two axes of ``x``
    (float32 or float64 CUDA tensors, even last dimension, ``k`` of shape x.shape[-2:])."""
    global _FN
    if _FN is None:
        _FN = _autograd_function()
    # where no backward pass is recorded nothing is kept for the gradient of k
    return _FN.apply(x, k, _torch().is_grad_enabled())


def FFTConvolve2D(H: int, W: int, dtype=None, init_std: float = 0.01):
    """``torch.nn.Module`` holding a learnable (H, W) kernel applied with ``fft_convolve2d``."""
    torch = _torch()

    class _M(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.kernel = torch.nn.Parameter(init_std * torch.randn(H, W, dtype=dtype or torch.float32,
                                                                    device="cuda"))

        def forward(self, x):
            return fft_convolve2d(x, self.kernel)

    return _M()
