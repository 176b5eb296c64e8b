"""
1-D conservative weights of short elements, of 24 to 48 vertices in all at the
most, in numbers around 4096: one thread sweeps each or a block takes it cell
by cell.  Bit for bit against the oracle.
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


@pytest.mark.parametrize("D,n,m", [(5, 2, 2), (5, 14, 10), (5, 14, 11), (5, 2, 22), (5, 22, 3),
                                   (4095, 13, 12), (4096, 13, 12), (4096, 27, 21),
                                   (4096, 27, 22), (4100, 2, 46), (4100, 47, 2)])
def test_short_elements_match_oracle(D, n, m):
    rng = np.random.default_rng(n * 100 + m)
    xi = np.sort(rng.uniform(-1, 1, (D, n)), axis=1)
    xo = np.sort(rng.uniform(-1.2, 1.1, (D, m)), axis=1)
    xi[::3] = xi[::3, ::-1]
    xo[::5] = xo[::5, ::-1]
    if n > 3:
        xi[1, 1] = xi[1, 2]  # repeated, unordered, NaN
        xi[2, [0, 3]] = xi[2, [3, 0]]
        xi[4, 2] = np.nan
    wi = rng.uniform(0.5, 2, (D, n - 1))
    with np.errstate(invalid="ignore"):
        got, off = _build(xi, xo, wi)
        for d in range(D):
            ref = oracle.coalesce(*oracle.conservative_1d(xi[d], xo[d], wi[d]))
            for g, r in zip(got, ref):
                assert np.array_equal(g[off[d]:off[d + 1]], r, equal_nan=True), d
