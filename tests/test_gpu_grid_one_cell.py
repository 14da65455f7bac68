"""The table gradient of points that share few cells (padding at one place, say): hits of one row
are summed over the lanes before they are added.  Oracle and tolerance of test_gpu_grid_scatter."""
import pytest
import torch

from neural3dstrokes_amd.gridencoder import GridEncoder
from test_gpu_grid_scatter import _check


@pytest.mark.gpu
@pytest.mark.parametrize('C', [1, 2, 4, 8])
@pytest.mark.parametrize('places', [1, 2, 40])
def test_points_in_few_cells(C, places, dev):
    g = torch.Generator().manual_seed(places)
    n = 4133
    x = torch.rand(places, 3, generator=g)[torch.arange(n) * places // n] + 1e-4 * torch.rand(n, 3, generator=g)
    x[n // 2:n // 2 + 700] = torch.rand(700, 3, generator=g)  # and some apart
    x = x.clamp(0, 1)
    enc = GridEncoder(num_levels=5, level_dim=C, base_resolution=12, desired_resolution=190, log2_hashmap_size=15)
    _check(x, enc.offsets.tolist(), C, enc.per_level_scale, 12, dev)
