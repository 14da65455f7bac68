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
