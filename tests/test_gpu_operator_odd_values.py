"""The stroke and compositing operators' sparse paths on values that no sensible scene holds:
they answer as the general paths do, and what is not finite stays visible."""
import pytest
import torch

from conftest import rel_err
from neural3dstrokes_amd.strokelib import backend
from test_gpu_operator_paths import CURVES, _backward, _case, _forward

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


def _odd(case, kind, sid):
    x, r, view, sp, cp, _ = case
    if kind == 'radius':
        r[:6] = torch.tensor([-0.05, 0.0, -0.0, NAN, INF, -INF])
    elif kind == 'point':
        x[0, 0], x[1, 1], x[2], x[3, 2] = NAN, INF, -INF, NAN
    elif kind == 'param':
        for i in range(sp.shape[1]):
            sp[i, i], sp[30 + i, i] = NAN, INF if i % 2 else -INF
    elif sid & 12:  # a zero scale, a negative one
        end = sp.shape[1] - 3 * bool(sid & 1) - 3 * bool(sid & 2)
        sp[5, end - 1], sp[11, end - 1] = 0.0, -0.1
        sp[9, end - (1 if sid & 4 else 3):end] = 0.0


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['radius', 'point', 'param', 'scale'])
@pytest.mark.parametrize('base', range(12))
def test_live_adjoint_passes_odd_values(base, kind, dev):
    """A stroke or point that is not finite makes the same gradients infinite or NaN as on the
    general path (which runs when a zero SDF gradient is given); the others agree within the
    tolerances of test_gpu_operator_paths."""
    for single in (False, True):
        case = _case(base, 0, 70, 4, 16, dev, single=single, seed=base)
        x, r, view, sp, cp, sid = case
        _odd(case, kind, sid)
        g = torch.Generator().manual_seed(1)
        up = (torch.randn(64, 70, generator=g).to(dev), torch.randn(64, 70, 3, generator=g).to(dev))
        none = torch.empty(0, device=dev)
        for isr in (False, True):
            alpha, color = torch.empty(64, 70, device=dev), torch.empty(64, 70, 3, device=dev)
            backend.stroke_forward(alpha, color, none, none, x, r, view, sp, cp, sid, 0, 1.0, False, isr)
            for exact in (True, False):
                got = _backward(case, 0, exact, isr, False, up, True, alpha)
                want = _backward(case, 0, exact, isr, True, up, True, alpha)
                for a, b in zip(got, want):
                    fin = torch.isfinite(b)
                    assert torch.equal(torch.isfinite(a), fin)
                    assert rel_err(a[fin], b[fin]) < (1e-4 if base in CURVES else 1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize('value', [NAN, INF])
@pytest.mark.parametrize('D', [1, 3])
def test_compositing_passes_odd_values(D, value, dev):
    """A transparent stroke with an infinite or NaN colour or density: alpha's gradients of the
    strokes in front of it are not finite, whether or not a chunk of 64 holds another alpha
    (one of 1e-30, which leaves every transmittance as it is)."""
    g = torch.Generator().manual_seed(D)
    N, S = 6, 256  # the chunks are strokes 192..255, 128..191, ...
    a = torch.zeros(N, S)
    a[:, [3, 70, 200]] = torch.rand(N, 3, generator=g) * 0.9
    c, dp = torch.rand(N, S, D, generator=g), torch.rand(S, generator=g)
    gd, gc = torch.randn(N, generator=g).to(dev), torch.randn(N, D, generator=g).to(dev)
    out = []
    for where in ('none', 'colour', 'density'):
        cc, dd = c.clone(), dp.clone()
        if where == 'colour':
            cc[2, 150, D - 1] = value
        elif where == 'density':
            dd[140] = value
        for tiny in (0.0, 1e-30):
            at = a.clone()
            at[:, 130] = tiny
            t = [v.to(dev) for v in (at, cc, dd)]
            for mode in ('exact', 'reference'):
                ga, gcol, gdp = torch.full((N, S), 9.0, device=dev), torch.zeros_like(t[1]), torch.zeros_like(t[2])
                backend.compose_backward(ga, gcol, gdp, gd, gc, *t, mode)
                out.append((where, tiny, ga.cpu()))
    for i in range(0, len(out), 4):
        for (where, _, x), (_, _, y) in zip(out[i:i + 2], out[i + 2:i + 4]):
            fin = torch.isfinite(y)
            assert torch.equal(torch.isfinite(x), fin) and rel_err(x[fin], y[fin]) < 1e-5
            assert bool(fin.all()) == (where == 'none')
            assert where == 'none' or not fin[2, 200]
