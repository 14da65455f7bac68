"""The split adjoint when its pool of record pages runs out, seen to happen: the rays left to the
one-kernel adjoint are read from the flags in the workspace.

Gradients against the one-kernel adjoint's within 1e-5, the float summation order (the tolerance
of the other split-adjoint tests)."""
import pytest
import torch

from conftest import rel_err
from neural3dstrokes_amd import render, scenes
from test_gpu_split_pool import _grads

MARK = 0x7fabcdef


@pytest.mark.gpu
@pytest.mark.parametrize('n_strokes', [60, 150])
def test_pool_runs_out(n_strokes, dev, monkeypatch):
    """16385 rays of 32 samples, one record per ray and family asked for: a wavefront's own page
    of a family holds 256 records, and there are 193 pages more for 4096 wavefronts."""
    R = 16385
    gen = torch.Generator().manual_seed(4)
    sc = scenes.make_strokes([0, 10] * (n_strokes // 2), gen, color_id=0)
    sc.update(scenes.make_rays(R, 32, gen, radius=0.004))
    kw = dict(use_laplace_transform=True, sdf_delta=2.0, cone=True, store=(n_strokes, 2048))
    spaces = []

    def workspace(floats, extra, device):
        spaces.append(torch.full((floats,), MARK, dtype=torch.int32, device=device))
        return spaces[-1].view(torch.float32)

    monkeypatch.setattr(render, '_workspace', workspace)
    got = _grads(sc, dev, True, 1, **kw)
    # the flags [R] follow the count of pages asked for; only they are R zeros and ones in a row
    # (the gradient rows, at most 150 strokes of 20 columns, are shorter)
    ws = spaces[0]
    bit = torch.cat([ws.new_zeros(1, dtype=torch.bool), (ws == 0) | (ws == 1), ws.new_zeros(1, dtype=torch.bool)])
    step = bit[1:].int() - bit[:-1].int()
    start, end = torch.nonzero(step == 1).flatten(), torch.nonzero(step == -1).flatten()
    runs = [(int(s), int(e)) for s, e in zip(start, end) if e - s >= R]
    assert len(runs) == 1
    s = runs[0][0]
    flagged, asked = int(ws[s:s + R].sum()), int(ws[s - 1])
    assert asked > 193  # more than there are beyond the wavefronts' own
    assert R // 100 < flagged < R - R // 100
    want = _grads(sc, dev, False, 1, **kw)
    for a, b in zip(got, want):
        assert torch.isfinite(a).all() and float(a.abs().sum()) > 0
        assert rel_err(a, b) < 1e-5
