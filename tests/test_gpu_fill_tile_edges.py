"""
``rg_fill_gauss_seidel_2d`` in tiles, at the edges of a tile's interior (36 rows
of 92 columns): one cell less, as many and one more, for one to three tiles an
axis, bit for bit against the oracle's sequential sweep.
"""

import numpy as np
import pytest

from oracle import oracle
from regridding_amd._lib import DeviceArray, check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(108, 91), (109, 92), (107, 93), (71, 183), (72, 184), (73, 185),
                                   (35, 275), (36, 276), (37, 277), (36, 368), (144, 93)])
@pytest.mark.parametrize("density", [0.05, 1.0])
def test_tile_edges_match_sequential_sweep(shape, density):
    r = np.random.default_rng(shape[0] * 1000 + shape[1])
    a = r.uniform(-1, 1, size=(2, *shape))
    where = r.uniform(size=a.shape) < density
    where[:, :: 35, :] = True
    where[:, :, 90:94] = True
    for iters in (3, 9, 20):
        da = DeviceArray.from_host(a)
        dw = DeviceArray.from_host(where.astype(np.uint8))
        check(lib().rg_fill_gauss_seidel_2d(da.ptr, dw.ptr, *a.shape, iters, 0))
        assert np.array_equal(da.to_host(), oracle.fill_gauss_seidel_2d(a, where, iters)), iters
