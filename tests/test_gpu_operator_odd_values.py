"""The stroke and compositing operators' sparse paths on values that no sensible scene holds:
they answer as the general paths do, and what is not finite stays visible."""
import pytest
import torch

from test_gpu_operator_paths import CURVES, _case, _forward

NAN, INF = float('nan'), float('inf')


@pytest.mark.gpu
@pytest.mark.parametrize('base', CURVES)
def test_curve_forward_odd_radii(base, dev):
    """With a radius that is not positive the transfer's slope changes its sign: a point far from
    the curve is inside.  Tolerances of test_gpu_operator_paths: the slope here is at most 10."""
    x, r, view, sp, cp, sid = _case(base, 0, 70, 4, 16, dev, seed=base)
    r[:8] = torch.tensor([-0.05, -0.3, 0.0, -0.0, NAN, INF, -INF, 2.0])
    a, _, _ = _forward(x, r, view, sp, cp, sid, 0, False)
    w, _, _ = _forward(x, r, view, sp, cp, sid, 0, True)
    assert torch.equal(torch.isnan(a), torch.isnan(w))
    assert ((a.nan_to_num() - w.nan_to_num()).abs() > 3e-5).sum() * 2000 <= a.numel()
    assert float(w[0].max()) > 0.9
