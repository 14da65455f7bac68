"""The split adjoint with float rows that nearly fill the LDS: only for many rays and not too many
strokes, with the one-kernel adjoint's gradients (1e-5, as test_gpu_pair_rows states)."""
import pytest

from neural3dstrokes_amd import _lib
from test_gpu_split import _check, _scene


@pytest.mark.gpu
def test_rule(dev):
    floats = _lib.lib().n3ds_render_backward_split_floats
    # 27 columns: rows past 7/8 of 160 KB from 1328 strokes, past all of it from 1518; 18 columns:
    # from 1992 and 2276
    for rays, strokes, shape, colour, split in (
            (4096, 1327, 14, 12, True), (4096, 1328, 14, 12, False), (16383, 1516, 14, 12, False),
            (16384, 1517, 14, 12, True), (16384, 1518, 14, 12, False), (64, 1991, 14, 3, True),
            (65536, 1992, 14, 3, False), (65536, 2275, 14, 3, False), (64, 1137, 14, 3, True)):
        assert (floats(rays, strokes, shape, colour) > 0) == split


@pytest.mark.gpu
@pytest.mark.parametrize('strokes', [1328, 1516])
def test_many_rays_of_full_rows(strokes, dev):
    _check(_scene(16384, 32, strokes, seed=7, color_id=1), dev, color_id=1)
