"""Weight gradients of the proposal head over many equal points: the sum's own error.

With every point the same, a gradient is N times one point's, each term as large as the next and
rounded the same way when it is added.  A float32 chain of 64 additions (256 points, 4 to a
matrix instruction) is off by at most 64 x 2^-24 = 3.8e-6 of the sum; the chains meet in doubles.
The point's own gradient in float32 (features, density, its derivative) is good to 1e-6."""
import pytest
import torch
import torch.nn.functional as F

from neural3dstrokes_amd import propfield


@pytest.mark.gpu
@pytest.mark.parametrize('kw', [dict(), dict(grid_level_dim=2)])
@pytest.mark.parametrize('n', [1 << 16, 1 << 24])
def test_weight_gradients_of_equal_points(n, kw, dev):
    torch.manual_seed(1)
    m = propfield.PropDensityField(grid_log2_hashmap_size=14, **kw).to(dev)
    m.encoder.embeddings.requires_grad_(False).fill_(0.3)
    x = torch.tensor([[0.31, -0.72, 0.45]], device=dev)
    up = 0.7123
    ps = list(m.density_layer.parameters())
    got = torch.autograd.grad(m(x.expand(n, 3))['density'], ps, torch.full((n,), up, device=dev))
    with torch.no_grad():
        f = m.encoder(m(x)['coord'], bound=1.0).double()
    d = [p.detach().double().requires_grad_(True) for p in ps]
    raw = F.relu(f @ d[0].t() + d[1]) @ d[2].t() + d[3]
    want = torch.autograd.grad(F.softplus(raw + m.density_bias), d, torch.full_like(raw, float(torch.tensor(up))))
    for a, b in zip(got, want):
        assert float((a.double() - n * b).abs().max()) <= 5e-6 * n * float(b.abs().max())
