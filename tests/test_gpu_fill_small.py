"""
``rg_fill_gauss_seidel_2d`` on slices of one row or column and on slices of a
few cells, around the sizes where a slice's workgroup grows (256 cells) and
where it no longer fits the LDS (8192): bit for bit against the oracle's
sequential sweep.
"""

import numpy as np
import pytest

from oracle import oracle
from regridding_amd._lib import DeviceArray, check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 1, 1), (3, 1, 2), (3, 2, 1), (2, 1, 3), (2, 3, 1), (2, 2, 2),
                                   (2, 1, 64), (2, 64, 1), (2, 1, 255), (2, 257, 1), (1, 1, 1000),
                                   (1, 1001, 1), (1, 1, 8191), (1, 8192, 1), (1, 1, 8193),
                                   (5, 3, 3), (5, 4, 5), (70, 8, 8), (3, 15, 17), (3, 16, 16),
                                   (3, 1, 256), (3, 2, 129), (3, 17, 16), (3, 9, 29)])
@pytest.mark.parametrize("density", [0.2, 1.0])
def test_small_slices_match_sequential_sweep(shape, density):
    r = np.random.default_rng(shape[1] * 1000 + shape[2])
    a = r.uniform(-1, 1, size=shape)
    where = r.uniform(size=shape) < density
    where[:, -1, -1] = True
    for iters in (1, 2, 5, 12):
        da = DeviceArray.from_host(a)
        dw = DeviceArray.from_host(where.astype(np.uint8))
        check(lib().rg_fill_gauss_seidel_2d(da.ptr, dw.ptr, *a.shape, iters, 0))
        with np.errstate(all="ignore"):
            want = oracle.fill_gauss_seidel_2d(a, where, iters)
        assert np.array_equal(da.to_host(), want, equal_nan=True), iters
