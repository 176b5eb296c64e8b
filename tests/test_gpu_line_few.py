"""
1-D conservative weights at the edges of which elements one thread sweeps (2 n
+ m up to 50 vertices, more with the number of elements up to 150; from 50000
elements (n + m) min(n, 12) up to 600), next to those taken cell by cell: bit
for bit against the oracle.
"""

import ctypes

import numpy as np
import pytest

from oracle import oracle
from regridding_amd._lib import DeviceArray, check, lib

pytestmark = pytest.mark.gpu


def _build(xi, xo, wi):
    (D, n), m, L = xi.shape, xo.shape[1], lib()
    dxi, dxo, dwi = (DeviceArray.from_host(np.ascontiguousarray(a)) for a in (xi, xo, wi))
    counts = DeviceArray.empty((D * (n - 1),), np.int32)
    offs = DeviceArray.empty((D * (n - 1) + 1,), np.int64)
    total = ctypes.c_int64()
    check(L.rg_conservative_1d_count(dxi.ptr, n, dxo.ptr, m, D, counts.ptr, offs.ptr,
                                     ctypes.byref(total), 0))
    T = total.value
    ii, io, w = (DeviceArray.empty((max(T, 1),), t) for t in (np.int64, np.int64, np.float64))
    check(L.rg_conservative_1d_emit(dxi.ptr, n, dxo.ptr, m, D, dwi.ptr, counts.ptr, offs.ptr,
                                    ii.ptr, io.ptr, w.ptr, 0))
    return [a.to_host()[:T] for a in (ii, io, w)], offs.to_host()[:: n - 1]


# 200 different elements, repeated to D in another order (the oracle sweeps 200)
@pytest.mark.parametrize("D,n,m", [(249, 20, 10), (249, 20, 11), (250, 20, 11), (250, 20, 12),
                                   (249, 2, 46), (249, 2, 47), (249, 24, 2), (249, 24, 3),
                                   (25000, 60, 30), (25000, 60, 31), (49999, 74, 2),
                                   (49999, 74, 3), (50000, 2, 298), (50000, 2, 299),
                                   (50000, 12, 38), (50000, 12, 39), (50000, 11, 43),
                                   (50000, 11, 44), (50000, 48, 2), (50000, 48, 3)])
def test_elements_at_the_edge_match_oracle(D, n, m):
    rng = np.random.default_rng(n * 1000 + m)
    xi = np.sort(rng.uniform(-1, 1, (200, n)), axis=1)
    xo = np.sort(rng.uniform(-1.2, 1.1, (200, m)), axis=1)
    xi[::3] = xi[::3, ::-1]
    xo[::5] = xo[::5, ::-1]
    if n > 3:
        xi[1, 1] = xi[1, 2]  # repeated, unordered, NaN
        xi[2, [0, 3]] = xi[2, [3, 0]]
        xi[4, 2] = np.nan
    wi = rng.uniform(0.5, 2, (200, n - 1))
    with np.errstate(invalid="ignore"):
        refs = [oracle.coalesce(*oracle.conservative_1d(*a)) for a in zip(xi, xo, wi)]
    pick = np.concatenate([np.arange(200), rng.integers(0, 200, D - 200)])
    got, off = _build(xi[pick], xo[pick], wi[pick])
    sizes = np.array([len(r[0]) for r in refs])[pick]
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(sizes)]))
    for g, k in zip(got, range(3)):
        ref = np.concatenate([refs[p][k] for p in pick])
        assert np.array_equal(g, ref, equal_nan=True), k
