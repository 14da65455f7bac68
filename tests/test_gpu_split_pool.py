"""The split adjoint's pool of record pages: rays that find it empty, and rays with more
hits than the pending list.

The same upstream gradients through the split adjoint and through the one-kernel
adjoint; parameter gradients within 1e-5, the float summation order of sums over
10^4 to 10^6 pairs of either sign (the tolerance of the other split-adjoint tests).
"""
import pytest
import torch

from conftest import rel_err
from neural3dstrokes_amd import autotune, render, scenes


def _grads(sc, dev, split, cap, **kw):
    old = autotune.current()
    try:
        autotune.set('bwd_split', int(split))
        autotune.set('split_cap', cap)
        g = torch.Generator().manual_seed(3)
        R = sc['tdist'].shape[0]
        up = (torch.randn(R, 3, generator=g).to(dev), torch.randn(R, generator=g).to(dev))
        params = [sc[k].to(dev).requires_grad_(True) for k in ('shape_params', 'color_params', 'density_params')]
        rays = [sc[k].to(dev) for k in ('origins', 'directions', 'viewdirs', 'radii', 'tdist')]
        rgb, acc, _ = render.render_strokes(*rays, sc['stroke_ids'], *params, **kw)
        return torch.autograd.grad((rgb, acc), params, up)
    finally:
        for k, v in old.items():
            autotune.set(k, v)


def _check(sc, dev, cap, **kw):
    for a, b in zip(_grads(sc, dev, True, cap, **kw), _grads(sc, dev, False, cap, **kw)):
        assert torch.isfinite(a).all() and float(a.abs().sum()) > 0
        assert rel_err(a, b) < 1e-5


@pytest.mark.gpu
def test_rays_past_the_pool(dev):
    """Sized for one record per ray and family (the 16 rays of a wavefront hold 40 times
    that), the pool runs out part of the way: the rest goes to the one-kernel adjoint."""
    _check(scenes.make_workload('palette500_65536x128', seed=6), dev, 1)


@pytest.mark.gpu
@pytest.mark.parametrize('n_rays,n_samples', [(300, 32), (65, 64), (64, 100)])
def test_many_hits_per_ray(dev, n_rays, n_samples):
    """Soft edges: most of 330 ellipsoids reach every ray (more than the 128 pending hits)."""
    gen = torch.Generator().manual_seed(9)
    sc = scenes.make_strokes([0] * 330, gen, color_id=2)
    sc.update(scenes.make_rays(n_rays, n_samples, gen, radius=0.004))
    kw = dict(color_id=2, use_laplace_transform=True, sdf_delta=4.0, cone=True, inv_scale_radius=True)
    cnt = torch.zeros(25, dtype=torch.int64, device=dev)
    with torch.no_grad():
        render.render_strokes(*[sc[k].to(dev) for k in ('origins', 'directions', 'viewdirs', 'radii', 'tdist')],
                              sc['stroke_ids'], *[sc[k].to(dev) for k in ('shape_params', 'color_params',
                                                                         'density_params')], counters=cnt, **kw)
    assert int(cnt[24]) > 128 * n_rays
    _check(sc, dev, 32, **kw)
