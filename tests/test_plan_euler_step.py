"""The plan of a whole Euler step: equal segments of at most 200 rows, halved where
they would be longer, that cover every row of every strip once; the plan of the other
schemes everywhere else."""

import numpy as np
import pytest

from tests.test_plan_step import STEP, plan

EULER_STEP = 19


@pytest.mark.parametrize("nx,ny,tile_rows,waves,halved", [
    (64, 64, 0, 4, False), (4096, 4096, 0, 4, False), (7000, 7000, 0, 4, False), (7300, 7300, 0, 4, True),
    (8192, 8192, 0, 4, True), (9500, 7000, 0, 3, True), (10000, 10000, 0, 4, True), (8192, 8192, 304, 4, False),
])
def test_long_segments_are_halved(nx, ny, tile_rows, waves, halved):
    euler, other = (plan(s, nx, ny, tile_rows, waves) for s in (EULER_STEP, STEP))
    if not halved:
        assert np.array_equal(euler, other)
        return
    rows = [p[p[:, 0] >= 0] for p in (euler, other)]
    assert rows[1][:, 2].max() > 200
    assert rows[0][:, 2].max() == (rows[1][:, 2].max() + 1) // 2
    cover = np.zeros((-(-nx // 56), ny), dtype=np.int8)
    for s, r, c in rows[0]:
        cover[s, r:r + c] += 1
    assert (cover == 1).all()
