"""Interval sampling with its bins in registers (by 64, up to 256) and above.

Appending bins of zero width and weight leaves the distribution as it is and moves it to the
next register count, or to none.  Only the closing of the CDF moves: 1 in place of a float32
sum of at most 300 terms, 300 * 2^-24 = 1.8e-5; in a last bin of weight 0.2 and width 0.1 a
centre moves by at most 1.8e-5 / 0.2 * 0.1 = 9e-6, and an end fencepost by three times that.
"""
import pytest
import torch

from neural3dstrokes_amd import stepfun


@pytest.mark.gpu
@pytest.mark.parametrize('m', [1, 2, 63, 64, 65, 128, 129, 192, 193, 256, 257])
@pytest.mark.parametrize('n', [2, 63, 64, 65, 128, 129, 200])
def test_padded_bins(m, n, dev):
    g = torch.Generator().manual_seed(m)
    R = 33
    t = torch.sort(torch.rand(R, m + 1, generator=g) * 0.9, -1).values
    t[:, -1] = t[:, -2] + 0.1
    w = torch.rand(R, m, generator=g) ** 3 + 1e-3
    w = w / w.sum(-1, keepdim=True) * 0.8
    w[:, -1] += 0.2
    lg = torch.log(w)
    want = stepfun.sample_intervals(False, t.to(dev), lg.to(dev), n, domain=(0.0, 2.0))
    # fenceposts lie in the bins and in order
    assert torch.isfinite(want).all() and (want[:, 1:] >= want[:, :-1]).all()
    for pad in (1, 64, 300 - m):
        tp = torch.cat([t, t[:, -1:].expand(R, pad)], 1).to(dev)
        lp = torch.cat([lg, torch.full((R, pad), -float('inf'))], 1).to(dev)
        got = stepfun.sample_intervals(False, tp, lp, n, domain=(0.0, 2.0))
        assert (got - want).abs().max() < 2.7e-5
