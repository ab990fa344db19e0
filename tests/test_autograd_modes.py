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
