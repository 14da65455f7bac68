"""Two half features in levels larger than the parts that single features are gathered in: taken
whole, with the one kernel's values to the bit (as test_gpu_prop_levels states them)."""
import pytest
import torch

from neural3dstrokes_amd.gridencoder import GridEncoder
from test_gpu_prop_levels import _forward


@pytest.mark.gpu
@pytest.mark.parametrize('n', [1 << 18, 600001])
def test_two_halves_in_large_levels(n, dev):
    torch.manual_seed(4)
    enc = GridEncoder(num_levels=10, level_dim=2, log2_hashmap_size=21, base_resolution=16,
                      desired_resolution=500).to(dev)
    off = enc.offsets.tolist()
    assert max(b - a for a, b in zip(off, off[1:])) * 4 > 4 << 20
    emb = (torch.rand(enc.embeddings.shape, device=dev) * 2 - 1).half()
    lin0, lin1 = torch.nn.Linear(20, 64).to(dev), torch.nn.Linear(64, 1).to(dev)
    x = torch.rand(n, 3, device=dev) * 2.4 - 1.2
    need, *a = _forward(enc, emb, x, lin0, lin1, 0, True)
    assert need == n * 20 * 4
    _, *b = _forward(enc, emb, x, lin0, lin1, 0, False)
    for s, t in zip(a, b):
        assert torch.equal(s.view(torch.int32), t.view(torch.int32))
