"""Differentiable FFT-convolution: the hand-written adjoint against FP64 central
finite differences (eps 1e-4, 64 seeded entries of each gradient), against
torch.fft autograd (FP64 and FP32), and against the FP64 oracle forward."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _fft_conv():
    from vkdispatch_amd.fft.autograd import fft_convolve2d
    return fft_convolve2d


def _torch_ref(x, k):
    H, W = x.shape[-2:]
    return torch.fft.irfft2(torch.fft.rfft2(x) * torch.conj(torch.fft.rfft2(k)), s=(H, W))


def _loss_np(x, k, t):
    y = O.convolve2DR(x, np.fft.rfft2(k), kernel_inner_only=True)
    return 0.5 * np.sum((y - t) ** 2)


def test_forward_matches_oracle_and_convolve2DR_semantics():
    f = _fft_conv()
    rng = np.random.default_rng(0)
    x = rng.standard_normal((3, 64, 48))
    k = 0.1 * rng.standard_normal((64, 48))
    for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 2e-6)):
        xt = torch.tensor(x, dtype=dtype, device="cuda")
        kt = torch.tensor(k, dtype=dtype, device="cuda")
        y = f(xt, kt).cpu().numpy()
        ref = O.convolve2DR(x, np.fft.rfft2(k), kernel_inner_only=True)
        assert O.rel_l2(y, ref) < tol
        # y[n] = sum_m x[n+m] k[m] (circular cross-correlation)
    small_x, small_k = x[:1, :6, :4], k[:6, :4]
    ys = f(torch.tensor(small_x, device="cuda"), torch.tensor(small_k, device="cuda")).cpu().numpy()
    assert np.allclose(ys, O.correlate_bruteforce(small_x, small_k).real)


def test_gradients_vs_fp64_central_differences():
    f = _fft_conv()
    rng = np.random.default_rng(1)
    B, H, W = 2, 32, 24
    x = rng.standard_normal((B, H, W))
    k = 0.01 * rng.standard_normal((H, W))
    t = rng.standard_normal((B, H, W))
    xt = torch.tensor(x, device="cuda", requires_grad=True)
    kt = torch.tensor(k, device="cuda", requires_grad=True)
    y = f(xt, kt)
    loss = 0.5 * ((y - torch.tensor(t, device="cuda")) ** 2).sum()
    loss.backward()
    dx = xt.grad.cpu().numpy()
    dk = kt.grad.cpu().numpy()
    eps = 1e-4
    for arr, grad, which in ((x, dx, "x"), (k, dk, "k")):
        flat = rng.choice(arr.size, size=64, replace=False)
        for idx in flat:
            pos = np.unravel_index(idx, arr.shape)
            ap, am = arr.copy(), arr.copy()
            ap[pos] += eps
            am[pos] -= eps
            if which == "x":
                fd = (_loss_np(ap, k, t) - _loss_np(am, k, t)) / (2 * eps)
            else:
                fd = (_loss_np(x, ap, t) - _loss_np(x, am, t)) / (2 * eps)
            assert abs(fd - grad[pos]) <= 1e-6 * max(1.0, abs(fd)), (which, pos, fd, grad[pos])


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-5)])
def test_gradients_vs_torch_fft_autograd(dtype, tol):
    f = _fft_conv()
    g = torch.Generator(device="cpu").manual_seed(2)
    x = torch.randn(4, 128, 96, generator=g, dtype=dtype).cuda()
    k = (0.01 * torch.randn(128, 96, generator=g, dtype=dtype)).cuda()
    t = torch.randn(4, 128, 96, generator=g, dtype=dtype).cuda()
    xa, ka = x.clone().requires_grad_(), k.clone().requires_grad_()
    xb, kb = x.clone().requires_grad_(), k.clone().requires_grad_()
    (0.5 * ((f(xa, ka) - t) ** 2).sum()).backward()
    x64, k64 = x.double().requires_grad_(), k.double().requires_grad_()
    (0.5 * ((_torch_ref(x64, k64) - t.double()) ** 2).sum()).backward()
    assert O.rel_l2(xa.grad.double().cpu().numpy(), x64.grad.cpu().numpy()) < tol
    assert O.rel_l2(ka.grad.double().cpu().numpy(), k64.grad.cpu().numpy()) < tol


def test_differentiable_convolution_32x1024x1024():
    """Batch 32 of float32 1024x1024 N(0,1) images, learnable 1024x1024 kernel N(0, 0.01),
    L = 0.5 ||y - t||^2 with t ~ N(0,1): gradients vs torch.fft autograd in FP64."""
    f = _fft_conv()
    g = torch.Generator(device="cpu").manual_seed(0)
    x = torch.randn(32, 1024, 1024, generator=g).cuda()
    k = (0.01 * torch.randn(1024, 1024, generator=g)).cuda()
    t = torch.randn(32, 1024, 1024, generator=g).cuda()
    xa, ka = x.clone().requires_grad_(), k.clone().requires_grad_()
    y = f(xa, ka)
    (0.5 * ((y - t) ** 2).sum()).backward()
    x64, k64 = x.double().requires_grad_(), k.double().requires_grad_()
    y64 = _torch_ref(x64, k64)
    (0.5 * ((y64 - t.double()) ** 2).sum()).backward()
    assert O.rel_l2(y.detach().double().cpu().numpy(), y64.detach().cpu().numpy()) < 1e-5
    assert O.rel_l2(xa.grad.double().cpu().numpy(), x64.grad.cpu().numpy()) < 1e-5
    assert O.rel_l2(ka.grad.double().cpu().numpy(), k64.grad.cpu().numpy()) < 1e-5


@pytest.mark.parametrize("shape,dtype", [((3, 64, 48), torch.float32), ((5, 210, 130), torch.float32), ((1, 32, 2), torch.float32),
                                         ((33, 128, 66), torch.float32), ((2, 1024, 34), torch.float32),
                                         ((2, 31, 30), torch.float32), ((9, 96, 1000), torch.float32),
                                         ((3, 64, 48), torch.float64), ((2, 512, 36), torch.float64)])
@pytest.mark.parametrize("which", ["both", "x", "k"])
def test_packed_columns_and_their_adjoint(shape, dtype, which):
    """Columns that do not fill a tile (24, 65, 33, 17 of them), one column only, one image,
    groups that end early (33 images), a height without a column tile (31): output and
    gradients against torch.fft in FP64.  FP32 bound: six FFT passes at 3e-7 and a sum."""
    g = torch.Generator().manual_seed(shape[1])
    x, gy = (torch.randn(shape, generator=g, dtype=torch.float64) for _ in range(2))
    k = torch.randn(shape[1:], generator=g, dtype=torch.float64)
    F = torch.fft
    X, K, G = F.rfft2(x.to(dtype).double()), F.rfft2(k.to(dtype).double()), F.rfft2(gy.to(dtype).double())
    want = {"y": F.irfft2(X * K.conj(), s=shape[1:]), "x": F.irfft2(G * K, s=shape[1:]),
            "k": F.irfft2((X * G.conj()).sum(0), s=shape[1:])}
    xd = x.to(dtype).cuda().requires_grad_(which != "k")
    kd = k.to(dtype).cuda().requires_grad_(which != "x")
    y = _fft_conv()(xd, kd)
    y.backward(gy.to(dtype).cuda())
    tol = 2e-6 if dtype is torch.float32 else 1e-13
    for name, got in (("y", y.detach()), ("x", xd.grad), ("k", kd.grad)):
        if got is None:
            assert which != "both" and name not in ("y", which)
            continue
        ref = want[name]
        assert float((got.cpu().double() - ref).norm() / ref.norm()) < tol, name


def test_nothing_is_kept_without_a_backward_pass(monkeypatch):
    """Under no_grad a learnable kernel takes the launch that stores no transforms."""
    from vkdispatch_amd.fft import autograd
    kept = []
    forward = autograd._forward
    monkeypatch.setattr(autograd, "_forward", lambda x, k, plans, keep=False: kept.append(keep) or
                        forward(x, k, plans, keep))
    x = torch.randn(2, 64, 48, device="cuda")
    k = torch.randn(64, 48, device="cuda", requires_grad=True)
    with torch.no_grad():
        y0 = _fft_conv()(x, k)
    y1 = _fft_conv()(x, k)
    assert kept == [False, True] and not y0.requires_grad and y1.requires_grad
    assert torch.equal(y0, y1.detach())
