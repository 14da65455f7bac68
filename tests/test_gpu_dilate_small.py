"""Weight dilation with at most 64 bins (one per lane) and above, edge by edge.

Every output is a sort, a clip, a maximum and single float32 operations: a float32
restatement gives the same bits.  Renormalised weights add a float32 sum of at most 192
non-negative terms (192 roundings of 2^-24: 2e-5 at most) and a division.
"""
import numpy as np
import pytest
import torch

from neural3dstrokes_amd import stepfun


def _restated(t, w, d, lo, hi):
    f = np.float32
    d, lo, hi, eps = f(d), f(lo), f(hi), np.finfo(f).eps
    p = w / np.maximum(t[:, 1:] - t[:, :-1], eps)
    b, c = t[:, :-1] - d, t[:, 1:] + d
    e = np.clip(np.sort(np.concatenate([t, b, c], 1), axis=1), lo, hi)
    x = e[:, :-1, None]
    inside = (b[:, None] <= x) & (c[:, None] > x)
    pd = np.where(inside.all(-1), f(-np.inf), f(0))
    pd = np.maximum(pd, np.where(inside, p[:, None], f(-np.inf)).max(-1))
    return e, pd * (e[:, 1:] - e[:, :-1])


@pytest.mark.gpu
@pytest.mark.parametrize('m', [1, 2, 31, 63, 64, 65])
@pytest.mark.parametrize('kind', ['plain', 'ties', 'wide', 'clipped', 'open', 'none', 'zero'])
def test_dilate(m, kind, dev):
    rng = np.random.default_rng(m)
    R = 517
    t = np.sort(rng.random((R, m + 1)).astype(np.float32), 1)
    w = rng.random((R, m)).astype(np.float32) ** 4
    d, dom = 0.005, (0.0, 1.0)
    if kind == 'ties':  # edges and their shifts on one lattice of exact values
        t, d = np.sort(rng.integers(0, 17, (R, m + 1)).astype(np.float32) / 16, 1), 0.125
    elif kind == 'wide':
        d = 0.7
    elif kind == 'clipped':
        dom = (0.25, 0.75)
    elif kind == 'open':
        dom = (-np.inf, np.inf)
    elif kind == 'none':
        d = 0.0
    elif kind == 'zero':
        w[::2] = 0
        t[::3] = t[::3, :1]
    tt, ww = torch.from_numpy(t).to(dev), torch.from_numpy(w).to(dev)
    e, x = stepfun.max_dilate_weights(tt, ww, d, domain=dom)
    re, rx = _restated(t, w, d, *dom)
    assert np.array_equal(e.cpu().numpy(), re)
    assert np.array_equal(x.cpu().numpy(), rx)
    _, y = stepfun.max_dilate_weights(tt, ww, d, domain=dom, renormalize=True)
    ry = rx.astype(np.float64)
    ry = ry / np.maximum(ry.sum(1, keepdims=True), np.finfo(np.float32).eps)
    assert np.allclose(y.cpu().numpy(), ry, rtol=3e-5, atol=0)


@pytest.mark.gpu
def test_unsorted_rays_keep_their_neighbours(dev):
    """A ray out of order goes its own way; the others of its block are as without it."""
    g = torch.Generator().manual_seed(1)
    t = torch.sort(torch.rand(64, 33, generator=g), -1).values.to(dev)
    w = torch.rand(64, 32, generator=g).to(dev)
    a = stepfun.max_dilate_weights(t, w, 0.01, domain=(0.0, 1.0))
    u = t.clone()
    u[5] = u[5].flip(0)
    u[6, 3] = float('nan')
    b = stepfun.max_dilate_weights(u, w, 0.01, domain=(0.0, 1.0))
    keep = [i for i in range(64) if i not in (5, 6)]
    for x, y in zip(a, b):
        assert torch.equal(x[keep], y[keep])
