"""
``rg_fill_gauss_seidel_2d`` on slices that span several tiles, bit for bit
against the oracle's sequential sweep: odd and even axes (the periodic wrap
joins cells of one colour at an odd one), axes shorter than a tile (which then
holds several periodic images), the edges of a tile's interior (60 cells) and
of the slices kept whole in LDS (8192 cells), iteration counts around a
launch's eight, dense, sparse and empty masks.
"""

import numpy as np
import pytest

from oracle import oracle
from regridding_amd._lib import DeviceArray, check, lib

pytestmark = pytest.mark.gpu


def _run(a, where, iters):
    da = DeviceArray.from_host(a)
    dw = DeviceArray.from_host(where.astype(np.uint8))
    check(lib().rg_fill_gauss_seidel_2d(da.ptr, dw.ptr, *a.shape, iters, 0))
    return da.to_host()


@pytest.mark.parametrize("shape", [(2, 64, 128), (1, 90, 91), (1, 91, 91), (1, 120, 180),
                                   (2, 121, 181), (1, 17, 601), (1, 601, 17), (1, 16, 700),
                                   (1, 19, 479), (1, 15, 800), (1, 119, 60 * 5 + 1)])
@pytest.mark.parametrize("density", [0.03, 1.0])
def test_tiles_match_sequential_sweep(shape, density):
    r = np.random.default_rng(shape[1] * 1000 + shape[2])
    a = r.uniform(-1, 1, size=shape)
    where = r.uniform(size=shape) < density
    where[:, -1, ::2] = True  # the odd edges' last row and column
    where[:, ::2, -1] = True
    for iters in (2, 3, 8, 17, 33):
        assert np.array_equal(_run(a, where, iters),
                              oracle.fill_gauss_seidel_2d(a, where, iters)), iters


def test_empty_mask_and_empty_tiles_leave_the_array():
    r = np.random.default_rng(1)
    a = r.uniform(-1, 1, size=(2, 200, 201))
    where = np.zeros(a.shape, bool)
    assert np.array_equal(_run(a, where, 20), a)
    where[1, 3:9, 5:20] = True
    assert np.array_equal(_run(a, where, 20), oracle.fill_gauss_seidel_2d(a, where, 20))
