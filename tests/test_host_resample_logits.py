"""The resampling logits of weights with gradients (plain torch, on the CPU)."""
import torch

from neural3dstrokes_amd import stepfun


def test_weights_changed_before_the_backward():
    s = torch.linspace(0, 1, 5)
    w = torch.tensor([0.1, 0.2, 0.3, 0.4], requires_grad=True)
    own = w * 1.0
    logits = stepfun.resample_logits(s, own)
    with torch.no_grad():
        own.mul_(2.0)
    logits.sum().backward()
    assert torch.allclose(w.grad, 1 / w.detach())


def test_slope_at_negative_zero():
    w = torch.tensor([-0.0, 0.5], requires_grad=True)
    stepfun.resample_logits(torch.linspace(0, 1, 3), w).sum().backward()
    assert w.grad[0] == float('inf') and w.grad[1] == 2.0


def test_passes_without_gradients():
    s, w = torch.tensor([0.0, 0.25, 0.25, 1.0]), torch.tensor([0.5, 0.5, -0.0])
    for ww in (w, w.clone().requires_grad_(True), w.double(), w.half()):
        got = stepfun.resample_logits(s, ww)
        assert got.dtype == (torch.float64 if ww.dtype == torch.float64 else torch.float32)
        assert got[1] == -float('inf') and got[2] == -float('inf') and torch.isclose(got[0].float(), w[0].log(), rtol=1e-3)
