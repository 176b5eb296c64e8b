"""
The exhaustive part of the cell search: points the secant iteration gives up
on, all of a call's (the grid's middle cell has no width, so the first step is
singular) or a run of them (NaN), for point counts around a block's and around
its growth, against the oracle.
"""

import numpy as np
import pytest

from oracle import oracle
from regridding_amd import workloads
from regridding_amd._lib import DeviceArray, check, lib

pytestmark = pytest.mark.gpu
OUTSIDE = np.iinfo(np.int64).max


def _search(grid, px, py):
    dx, dy, dpx, dpy = (DeviceArray.from_host(np.ascontiguousarray(a)) for a in (*grid, px, py))
    out = DeviceArray.empty((px.size, 2), np.int64)
    check(lib().rg_find_cells_2d(dx.ptr, dy.ptr, *grid[0].shape, dpx.ptr, dpy.ptr, px.size,
                                 out.ptr, 0))
    return out.to_host()


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 500, 2000])
def test_every_point_searched_exhaustively(n):
    x, y = (a.copy() for a in workloads.warped_grid((9, 8), 0.3, 0.05, 0.04))
    x[5], y[5] = x[4], y[4]  # cells (4, j) have no width
    p = np.random.default_rng(n).uniform(-1.3, 1.3, (2, n))
    got = _search((x, y), *p)
    want = [oracle.index_of_point_secant((p[0, q], p[1, q]), (x, y)) for q in range(n)]
    assert np.array_equal(got, np.array(want).reshape(n, 2))
    assert n < 500 or 0 < (got[:, 0] != OUTSIDE).sum() < n


# (wavefronts look at 1, 2 and 64 points each)
@pytest.mark.parametrize("n,run", [(32767, 3000), (32768, 3000), (65537, 5000), (2097159, 9000)])
def test_a_run_of_points_without_a_cell(n, run):
    grid = workloads.warped_grid((41, 37), 0.3, 0.05, 0.04)
    p = np.random.default_rng(n).uniform(-1.2, 1.2, (2, n))
    want = _search(grid, *p)
    assert 0 < (want[:, 0] != OUTSIDE).sum() < n
    for at in (0, n // 2, n - run):
        q = p.copy()
        q[0, at:at + run] = np.nan
        got = _search(grid, *q)
        assert np.all(got[at:at + run] == OUTSIDE)
        got[at:at + run] = want[at:at + run]
        assert np.array_equal(got, want)
