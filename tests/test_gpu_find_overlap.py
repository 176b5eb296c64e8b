"""
Cell searches that overlap on one GPU, on streams of their own, with points
that need the exhaustive search (NaN among them): each gets its own result,
with ``rg_find_cells_2d_noalloc`` as with ``rg_find_cells_2d``.
"""

import numpy as np
import pytest
import torch

from regridding_amd import workloads
from regridding_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _search(fn, grid, points, stream):
    (x, y), (px, py) = grid, points
    ij = torch.empty((px.numel(), 2), dtype=torch.int64, device="cuda")
    check(fn(x.data_ptr(), y.data_ptr(), *x.shape, px.data_ptr(), py.data_ptr(), px.numel(),
             ij.data_ptr(), stream))
    return ij


@pytest.mark.parametrize("name", ["rg_find_cells_2d", "rg_find_cells_2d_noalloc"])
def test_overlapping_searches(name):
    L = lib()
    grids, points = [], []
    for k in range(4):
        g = workloads.warped_grid(41, 0.1 + 0.2 * k, 0.05, 0.04)
        p = np.random.default_rng(k).uniform(-1, 1, (2, 60000))
        p[:, k::97] = np.nan
        grids.append([torch.as_tensor(np.ascontiguousarray(a), device="cuda") for a in g])
        points.append([torch.as_tensor(a, device="cuda") for a in p])
    want = [_search(L.rg_find_cells_2d, g, p, 0) for g, p in zip(grids, points)]
    streams = [torch.cuda.Stream() for _ in grids]
    torch.cuda.synchronize()
    for _ in range(5):
        got = [_search(getattr(L, name), g, p, s.cuda_stream)
               for g, p, s in zip(grids, points, streams)]
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
