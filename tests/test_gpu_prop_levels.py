"""Proposal features gathered level by level (large tables, many points) against the one kernel.

Both sum a feature's 8 products in the same order with the same operations: equal to the bit,
and so are the densities and the warped coordinates.
"""
import numpy as np
import pytest
import torch

from neural3dstrokes_amd import _lib
from neural3dstrokes_amd.gridencoder import GridEncoder


def _forward(enc, emb, x, lin0, lin1, warp, workspace):
    lib, N, L, C = _lib.lib(), x.shape[0], enc.num_levels, enc.level_dim
    F, flag = L * C, int(emb.dtype == torch.half)
    d, co = torch.full((N,), 7.0, device=x.device), torch.empty(N, 3, device=x.device)
    f, x01 = torch.full((N, F), 7.0, device=x.device), torch.empty(N, 3, device=x.device)
    need = lib.n3ds_prop_field_workspace_bytes(N, L, C, emb.shape[0], flag)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=x.device) if workspace else None
    w1, b1, w2, b2 = (t.detach() for t in (lin0.weight, lin0.bias, lin1.weight, lin1.bias))
    _lib.check(lib.n3ds_prop_field_forward_ws(
        _lib.ptr(x), N, warp, 4.0, _lib.ptr(emb), _lib.ptr(enc.offsets), L, C, float(np.log2(enc.per_level_scale)),
        int(enc.base_resolution), enc.gridtype_id, int(enc.align_corners), enc.interp_id, flag, _lib.ptr(w1),
        _lib.ptr(b1), _lib.ptr(w2), _lib.ptr(b2), -1.0, _lib.ptr(d), _lib.ptr(co), _lib.ptr(f), _lib.ptr(x01),
        emb.shape[0], _lib.ptr(ws), need if workspace else 0, _lib.stream()))
    return need, d, co, f, x01


@pytest.mark.gpu
@pytest.mark.parametrize('n', [1 << 18, (1 << 18) + 1, 600001, (1 << 22) + 5])
@pytest.mark.parametrize('kind', ['float', 'half', 'half2', 'smooth', 'align', 'tiled', 'odd_rows', 'shifted'])
def test_levels_match_one_kernel(kind, n, dev):
    if n > 600001 and kind not in ('float', 'half2'):
        pytest.skip('the chunks do not depend on the rows')
    kw = dict(num_levels=10, level_dim=1, log2_hashmap_size=20)
    kw.update({'float': dict(log2_hashmap_size=22), 'half': dict(log2_hashmap_size=23),
               'half2': dict(level_dim=2), 'smooth': dict(interpolation='smoothstep'),
               'align': dict(align_corners=True), 'tiled': dict(gridtype='tiled')}.get(kind, {}))
    torch.manual_seed(3)
    enc = GridEncoder(**kw).to(dev)
    if kind == 'odd_rows':  # hashed levels of a row count that is no power of 2, and an empty one
        off = enc.offsets.cpu().numpy().copy()
        off[6:] -= 24
        off[8] = off[7]
        enc.offsets = torch.from_numpy(off).to(dev)
    emb = torch.rand(enc.embeddings.shape, device=dev) * 2 - 1
    if kind == 'shifted':  # a table that starts 4 bytes past 16
        emb = torch.cat([emb.flatten()[:1], emb.flatten()])[1:].reshape(emb.shape)
        assert emb.data_ptr() % 16 == 4
    if kind in ('half', 'half2'):
        emb = emb.half()
    lin0, lin1 = torch.nn.Linear(10 * enc.level_dim, 64).to(dev), torch.nn.Linear(64, 1).to(dev)
    x = torch.rand(n, 3, device=dev) * 2.4 - 1.2  # some outside the grid
    x[5], x[70], x[71] = 1.0, -1.0, float('nan')
    need, *a = _forward(enc, emb, x, lin0, lin1, 0, True)
    assert need == min(n, 1 << 22) * 10 * enc.level_dim * 4
    _, *b = _forward(enc, emb, x, lin0, lin1, 0, False)
    for s, t in zip(a, b):
        assert torch.equal(s.view(torch.int32), t.view(torch.int32))


def test_level_rule():
    lib = _lib.lib()
    big = 1 << 22
    assert lib.n3ds_prop_field_workspace_bytes(1 << 18, 10, 1, big, 0) == (1 << 18) * 40
    assert lib.n3ds_prop_field_workspace_bytes(1 << 18, 10, 2, big, 1) == (1 << 18) * 80
    for args in (((1 << 18) - 1, 10, 1, big, 0), (1 << 18, 10, 2, (10 << 20) + 1, 1), (1 << 18, 10, 2, big, 0), (1 << 18, 8, 4, big, 1),
                 (1 << 18, 10, 1, 1 << 20, 0), (0, 10, 1, big, 0), (1 << 18, 0, 1, big, 0)):
        assert lib.n3ds_prop_field_workspace_bytes(*args) == 0
