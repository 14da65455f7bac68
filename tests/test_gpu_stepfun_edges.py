"""Weight dilation and interval sampling at the sizes where a lane takes one more edge or sample:
edges and single float32 operations to the bit, as test_gpu_dilate_small states them."""
import numpy as np
import pytest
import torch

from neural3dstrokes_amd import stepfun
from test_gpu_dilate_small import _restated


@pytest.mark.gpu
@pytest.mark.parametrize('m', [21, 22, 23])
def test_dilate_around_one_round_of_lanes(m, dev):
    rng = np.random.default_rng(m)
    t = np.sort(rng.integers(0, 40, (301, m + 1)).astype(np.float32) / 32, 1)
    w = rng.random((301, m)).astype(np.float32)
    for d, dom in ((0.125, (0.0, 1.0)), (0.01, (0.25, 0.75))):
        e, x = stepfun.max_dilate_weights(torch.from_numpy(t).to(dev), torch.from_numpy(w).to(dev), d, domain=dom)
        re, rx = _restated(t, w, d, *dom)
        assert np.array_equal(e.cpu().numpy(), re) and np.array_equal(x.cpu().numpy(), rx)


@pytest.mark.gpu
@pytest.mark.parametrize('m', [5, 64, 200, 256, 257, 400])
@pytest.mark.parametrize('n', [2, 64, 65, 128, 129, 193])
def test_sampling_keeps_positions(m, n, dev):
    """Bins of equal weight and width: the CDF is a ladder of m roundings of 2^-24 and its inverse
    the identity, so a centre is off by at most (m + 4) 2^-24 and an end by three times that."""
    t = torch.linspace(0, 1, m + 1, device=dev).expand(7, m + 1).contiguous()
    got = stepfun.sample_intervals(False, t, torch.zeros(7, m, device=dev), n, domain=(0.0, 1.0)).cpu().double()
    c = torch.linspace(1 / (2 * n), 1 - 1 / (2 * n) - np.finfo(np.float32).eps, n, dtype=torch.float64)
    mid = (c[1:] + c[:-1]) / 2
    want = torch.cat([(2 * c[:1] - mid[:1]).clamp_min(0), mid, (2 * c[-1:] - mid[-1:]).clamp_max(1)])
    assert (got - want).abs().max() <= 3 * (m + 4) * 2.0 ** -24
