"""The stroke adjoint's gradient to the points where most pairs are live: runs of one point's
entries as long as a wavefront, shorter than it, and across its edges.

Against the same kernel on one stroke at a time, whose pairs are each a run of their own: the
same terms in another order, so a point's sum over S strokes is off by at most S roundings of
6e-8 of the sum of the terms' sizes."""
import pytest
import torch

from neural3dstrokes_amd.strokelib import backend
from test_gpu_operator_paths import CURVES, _backward, _case


@pytest.mark.gpu
@pytest.mark.parametrize('base', range(12))
def test_point_gradients_of_dense_pairs(base, dev):
    for n_str, n_rays, m in ((5, 10, 31), (64, 3, 17), (130, 5, 40)):
        case = _case(base, 0, n_str, n_rays, m, dev, seed=base, radius=3.0)
        x, r, view, sp, cp, sid = case
        N = x.shape[0]
        g = torch.Generator().manual_seed(2)
        up = (torch.randn(N, n_str, generator=g).to(dev), torch.zeros(N, n_str, 3, device=dev))
        alpha, color = torch.empty(N, n_str, device=dev), torch.empty(N, n_str, 3, device=dev)
        none = torch.empty(0, device=dev)
        backend.stroke_forward(alpha, color, none, none, x, r, view, sp, cp, sid, 0, 1.0, False, False)
        assert base not in CURVES or float(((alpha > 0) & (alpha < 0.9999)).float().mean()) > 0.9
        got = _backward(case, 0, True, False, False, up, True, alpha)[2]
        want, size = torch.zeros(N, 3, dtype=torch.float64, device=dev), torch.zeros(N, 3, device=dev)
        for s in range(n_str):
            one = (x, r, view, sp[s:s + 1], cp[s:s + 1], sid)
            part = _backward(one, 0, True, False, False, [u[:, s:s + 1].contiguous() for u in up], True,
                             alpha[:, s:s + 1].contiguous())[2]
            want += part
            size += part.abs()
        assert float(want.abs().sum()) > 0
        assert ((got - want).abs() <= n_str * 6e-8 * size).all()
