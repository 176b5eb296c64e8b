"""
The cell search the kernels run (secant_search: every vertex read once, cells
clearly beside the point rejected before the winding sum) against the
statement-by-statement one (index_secant) on the CPU: points inside, outside,
on vertices, on edges and their floating-point neighbours, on warped, folded,
degenerate and tiny grids and grids with NaN.
"""

import numpy as np
import pytest

from regridding_amd import workloads
from tests.test_emu_secant_xy import _pair


def _points(x, y, rng):
    """Random points, vertices, edge midpoints and centres, each also moved
    by one unit in the last place along either axis."""
    lo, hi = np.nanmin(x) - 0.2, np.nanmax(x) + 0.2
    px = [rng.uniform(lo, hi, 600), x.ravel(), (x[1:] + x[:-1]).ravel() / 2,
          (x[:, 1:] + x[:, :-1]).ravel() / 2, (x[1:, 1:] + x[:-1, :-1]).ravel() / 2]
    py = [rng.uniform(np.nanmin(y) - 0.2, np.nanmax(y) + 0.2, 600), y.ravel(),
          (y[1:] + y[:-1]).ravel() / 2, (y[:, 1:] + y[:, :-1]).ravel() / 2,
          (y[1:, 1:] + y[:-1, :-1]).ravel() / 2]
    px, py = np.concatenate(px), np.concatenate(py)
    ok = ~(np.isnan(px) | np.isnan(py))
    px, py = px[ok], py[ok]
    out_x, out_y = [px], [py]
    for d in (-np.inf, np.inf):
        out_x += [np.nextafter(px, d), px]
        out_y += [py, np.nextafter(py, d)]
    return np.concatenate(out_x), np.concatenate(out_y)


def _grids():
    yield "warped", workloads.warped_grid((23, 31), 0.3, 0.06, 0.04)
    yield "rectilinear", workloads.warped_grid((17, 14), 0.0, 0.0, 0.0)
    yield "rotated_90", workloads.warped_grid((12, 9), np.pi / 2, 0.0, 0.0)
    yield "two_by_two", workloads.warped_grid(2, 0.4, 0.0, 0.0)
    yield "thin", workloads.warped_grid((2, 20), 0.2, 0.02, 0.01)
    yield "folded", workloads.warped_grid((25, 25), 0.3, 0.6, 0.5)
    x, y = workloads.warped_grid((15, 13), 0.2, 0.02, 0.02)
    x, y = x.copy(), y.copy()
    x[5, 6], y[8, 3] = np.nan, np.nan
    yield "nan", (x, y)
    x, y = workloads.warped_grid((12, 12), 0.1, 0.02, 0.02)
    yield "collapsed", (x, np.zeros_like(y))
    for name, f in (("small", 1e-160), ("large", 1e160)):
        yield name, tuple(f * a for a in workloads.warped_grid((9, 9), 0.3, 0.05, 0.05))


@pytest.mark.parametrize("name", [n for n, _ in _grids()])
def test_search_equals_reference_form(name):
    x, y = dict(_grids())[name]
    px, py = _points(x, y, np.random.default_rng(3))
    a, b = _pair(x, y, px, py)
    assert np.array_equal(a, b)
