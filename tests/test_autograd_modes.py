"""The differentiable convolution under autograd's modes, on the CPU: the kernels are left out."""
import pytest

from vkdispatch_amd.fft import autograd

torch = pytest.importorskip("torch")
fwd_ad = torch.autograd.forward_ad


@pytest.fixture
def kept(monkeypatch):
    """Whether each call keeps what the gradient of k needs; the convolution returns x."""
    got = []

    def run(fn, x, k, plans, *rest):
        got.append(bool(rest[0]))
        return x.clone(), k.clone(), x.clone() if rest[0] else None
    monkeypatch.setattr(autograd, "_run", run)
    monkeypatch.setattr(autograd, "plans_for", lambda *a: None)
    return got


def test_what_is_kept(kept):
    x, k = torch.ones(2, 4, 4), torch.ones(4, 4, requires_grad=True)
    autograd.fft_convolve2d(x, k)
    with torch.no_grad():
        autograd.fft_convolve2d(x, k)
    autograd.fft_convolve2d(x, k.detach())
    assert kept == [True, False, False]


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("recorded", [True, False])
def test_forward_mode_is_refused(kept, which, recorded):
    """No tangent is dropped in silence, with or without recording."""
    args = [torch.ones(2, 4, 4), torch.ones(4, 4)]
    with fwd_ad.dual_level(), torch.set_grad_enabled(recorded):
        args[which] = fwd_ad.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises(NotImplementedError):
            autograd.fft_convolve2d(*args)


def test_launches_that_spill_have_one_that_does_not(monkeypatch):
    """plans_for compiles the launches that do all of the work; where one that does a part of it
    would spill, theirs take its place."""
    from vkdispatch_amd import dtypes as dt
    from vkdispatch_amd.buffer import Buffer
    from vkdispatch_amd.fft.kernels import SpillError
    plan = autograd._HalfPlans(2, 64, 48, dt.complex64)
    ran, spilling = [], set()

    def check(kernel):
        if kernel in spilling:
            raise SpillError(kernel.name)
    monkeypatch.setattr(autograd, "check_no_spill", check)
    monkeypatch.setattr(autograd, "_wrap", lambda t, var_type: Buffer(tuple(t.shape), var_type, (t.data_ptr(), t, True)))
    for name in ("conv", "conv_keep", "conv_dx", "grad", "rows_inv"):
        monkeypatch.setattr(getattr(plan, name), "launch", lambda v, name=name: ran.append((name, v)))
    x = torch.zeros(2, 64, 48)
    ws = autograd._wrap(autograd._spectra(plan, 2, "cpu"), plan.ctype)
    plan.forward(x, ws, ws, False)
    plan.backward(None, ws, x, ws, True, False)
    assert [n for n, _ in ran] == ["conv", "conv_dx", "rows_inv"]
    plan._fits.clear()
    ran.clear()
    spilling |= {plan.conv, plan.conv_dx}
    assert plan.forward(x, ws, ws, False) is None
    dx, dk = plan.backward(None, ws, x, ws, True, False)
    assert [n for n, _ in ran] == ["conv_keep", "grad", "rows_inv"] and dk is None and dx.shape == x.shape
    assert len(ran[0][1]) == 3 and ran[1][1][1] is ws and ran[1][1][3].size == plan.grad.groups * 64 * 24
