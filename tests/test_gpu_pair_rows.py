"""The pair kernel's rows: doubles while they fit the LDS, floats above, no split beyond.

The split adjoint against the one-kernel adjoint at stroke counts on both sides of either
line (18 columns: 1137 strokes in doubles, 2275 in floats; 27 columns with gradient_rgb: 758
and 1516).  The two differ in the order of float32 sums of at most a few thousand terms:
1e-5 of the largest entry, as for the other comparisons of these two.
"""
import pytest

from test_gpu_split import _check, _scene


@pytest.mark.gpu
@pytest.mark.parametrize('strokes,color_id', [(1, 0), (64, 0), (1137, 0), (1138, 0), (2275, 0), (2276, 0), (758, 1),
                                              (759, 1), (1516, 1), (1517, 1)])
def test_pair_rows(strokes, color_id, dev):
    _check(_scene(256, 64, strokes, seed=60 + strokes % 7, color_id=color_id), dev,
           **(dict(color_id=color_id) if color_id else {}))
