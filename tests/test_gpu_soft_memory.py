"""Memory of a training step with the Laplace transfer: what is kept for the backward and the
room for its records stay within their budget and the caller's capacities, and a step that fits
without the extra room does not run out of memory for it.

Gradients of the same step differ by the float summation order only: 1e-5, the tolerance of the
split-adjoint tests."""
import pytest
import torch

from conftest import rel_err
from neural3dstrokes_amd import _lib, render, scenes

MB = 1 << 20


def test_records_within_the_budget():
    b = render.STORE_BUDGET_BYTES
    assert render._split_records(65536, 128, False, 4096, 0) == 0
    for R, n, cap_p, kept in ((65536, 128, 4096, 1 << 30), (65536, 128, 4096, b - 512), (640000, 192, 1536, b),
                              (640000, 192, 1536, 2 * b), (4096, 64, 8, 1 << 20), (1, 1, 1, 0)):
        floats = render._split_records(R, n, True, cap_p, kept)
        assert 0 <= floats * 4 <= max(0, b - kept) and floats <= R * cap_p * 8
    assert render._split_records(16384, 32, True, 1024, 1 << 30) == 16384 * 32 * 16 * 8


def _step(dev, n_rays, n, store, **kw):
    gen = torch.Generator().manual_seed(2)
    sc = scenes.make_strokes([0] * 60, gen, color_id=0)
    sc.update(scenes.make_rays(n_rays, n, gen, radius=0.004))
    params = [sc[k].to(dev).requires_grad_(True) for k in ('shape_params', 'color_params', 'density_params')]
    rays = [sc[k].to(dev) for k in ('origins', 'directions', 'viewdirs', 'radii', 'tdist')]
    up = torch.randn(n_rays, 3, generator=gen).to(dev)
    rgb, _, _ = render.render_strokes(*rays, sc['stroke_ids'], *params, use_laplace_transform=True, sdf_delta=2.0,
                                      cone=True, store=store, **kw)
    return rgb, params, up, (len(sc['stroke_ids']), sc['shape_params'].shape[1], sc['color_params'].shape[1])


def _peak(rgb, params, up):
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    grads = torch.autograd.grad(rgb, params, up)
    torch.cuda.synchronize()
    return grads, torch.cuda.max_memory_allocated() - before


@pytest.mark.gpu
def test_capacities_bound_the_records(dev):
    """(cap_hits, cap_pairs) given by the caller: at most cap_pairs records a ray beyond the default."""
    R, n = 8192, 64
    rgb, params, up, (S, P, Q) = _step(dev, R, n, (8, 16))
    _, peak = _peak(rgb, params, up)
    least = 4 * max(_lib.lib().n3ds_render_backward_split_floats(R, S, P, Q),
                    _lib.lib().n3ds_render_backward_workspace_floats(R, S, P, Q))
    assert peak <= least + R * 16 * 32 + 4 * MB


@pytest.mark.gpu
def test_budget_bounds_the_records(dev, monkeypatch):
    R, n = 8192, 64
    monkeypatch.setattr(render, 'STORE_BUDGET_BYTES', 96 * MB)
    torch.cuda.synchronize()
    rgb, params, up, (S, P, Q) = _step(dev, R, n, 'auto')
    kept = render.keep_capacities(R, n, S, 0, True)[4]
    assert kept < 96 * MB
    _, peak = _peak(rgb, params, up)
    least = 4 * max(_lib.lib().n3ds_render_backward_split_floats(R, S, P, Q),
                    _lib.lib().n3ds_render_backward_workspace_floats(R, S, P, Q))
    assert peak <= least + (96 * MB - kept) + 4 * MB


@pytest.mark.gpu
def test_step_without_memory_for_the_records(dev):
    """torch's own limit leaves the default workspace, not the records: 32768 rays x 64 samples ask
    for 1 GiB more."""
    R, n = 32768, 64
    rgb, params, up, _ = _step(dev, R, n, True)
    want = torch.autograd.grad(rgb, params, up)
    del rgb
    rgb, params, up, (S, P, Q) = _step(dev, R, n, True)
    least = 4 * max(_lib.lib().n3ds_render_backward_split_floats(R, S, P, Q),
                    _lib.lib().n3ds_render_backward_workspace_floats(R, S, P, Q))
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + least + 256 * MB) / total)
        got = torch.autograd.grad(rgb, params, up)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for a, b in zip(got, want):
        assert rel_err(a, b) < 1e-5
