"""Box statistics behind the automatic depth: whole numbers, against a count on
the host, for repeated calls on one handle (the counts are left cleared)."""
import numpy as np
import pytest

import old_fmm_bem_amd as F


def _want(x):
    c = np.clip((x.astype(np.float32) * np.float32(256)).astype(np.int64), 0, 255)
    boxes, sumsq = np.zeros(9, np.int64), np.zeros(9)
    for l in range(9):
        s = c >> (8 - l)
        n = np.unique((s[:, 0] << 40) | (s[:, 1] << 20) | s[:, 2], return_counts=True)[1]
        boxes[l], sumsq[l] = len(n), float((n.astype(np.int64) ** 2).sum())
    return boxes, sumsq


# one point, every cell corner region, one cell, a surface, more points than cells of a level
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 1000, 70001])
def test_statistics_of_repeated_calls(n):
    rng = np.random.default_rng(n)
    cube = rng.random((n, 3))
    d = rng.standard_normal((n, 3))
    sets = [cube, 0.5 + 0.45 * d / np.linalg.norm(d, axis=1, keepdims=True), 0.3 + 1e-4 * cube,
            np.round(cube) * 0.999, cube]
    f = F.FMM(p=6, precision="mixed", convention="exact", box=(0, 0, 0, 1))
    for k, x in enumerate(sets):
        print(n, k, flush=True)
        x = x.astype(np.float32)
        f.set_points(x)
        boxes, sumsq = f.occupancy()
        wb, ws = _want(x)
        assert np.array_equal(boxes, wb) and np.array_equal(sumsq, ws)
    f.close()
