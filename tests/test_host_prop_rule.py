"""Where the proposal features are gathered level by level: ten levels, or eight and more that
stay in an L2, for enough points."""
import pytest

from neural3dstrokes_amd import _lib

MB = 1 << 20


@pytest.mark.parametrize('n,levels,dim,rows,half,staged', [
    (MB, 8, 1, 3 * MB, 0, True), (MB, 16, 1, 7 * MB, 0, True), (4 * MB + 1, 12, 1, 10 * MB, 1, True),
    (MB - 1, 8, 1, 3 * MB, 0, False),       # too few points
    (4 * MB, 7, 1, 3 * MB, 0, False),       # too few levels
    (4 * MB, 8, 1, 4 * MB, 0, False),       # levels of 2 MB on average: some are larger
    (4 * MB, 9, 2, 3 * MB, 1, False),       # two features
    (1 << 18, 10, 1, 14 * MB, 0, True), (1 << 18, 10, 2, 10 * MB, 1, True)])
def test_level_by_level_rule(n, levels, dim, rows, half, staged):
    got = _lib.lib().n3ds_prop_field_workspace_bytes(n, levels, dim, rows, half)
    assert got == (min(n, 4 * MB) * levels * dim * 4 if staged else 0)
