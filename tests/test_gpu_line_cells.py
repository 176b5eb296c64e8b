"""
The 1-D conservative sweep with one thread per input cell, at the edges of
its blocks (1024 cells) and searches (16 vertices), of the output vertices it
stages (2048) and of what it takes: an element with repeated or unordered
vertices or NaN goes through the serial sweep, beside monotonic elements of
the same call.  Bit for bit against the oracle through the C ABI.
"""

import ctypes

import numpy as np
import pytest

from oracle import oracle
from regridding_amd._lib import DeviceArray, check, lib

pytestmark = pytest.mark.gpu


def _build(xi, xo, wi):
    (D, n), m, L = xi.shape, xo.shape[1], lib()
    dxi, dxo = DeviceArray.from_host(xi), DeviceArray.from_host(xo)
    dwi = DeviceArray.from_host(wi) if wi is not None else None
    counts = DeviceArray.empty((D * (n - 1),), np.int32)
    offs = DeviceArray.empty((D * (n - 1) + 1,), np.int64)
    total = ctypes.c_int64()
    check(L.rg_conservative_1d_count(dxi.ptr, n, dxo.ptr, m, D, counts.ptr, offs.ptr,
                                     ctypes.byref(total), 0))
    T = total.value
    ii, io, w = (DeviceArray.empty((max(T, 1),), t) for t in (np.int64, np.int64, np.float64))
    check(L.rg_conservative_1d_emit(dxi.ptr, n, dxo.ptr, m, D, dwi.ptr if dwi else None,
                                    counts.ptr, offs.ptr, ii.ptr, io.ptr, w.ptr, 0))
    return [a.to_host()[:T] for a in (ii, io, w)], offs.to_host()[:: n - 1]


def _check(xi, xo, wi=None):
    got, off = _build(np.ascontiguousarray(xi), np.ascontiguousarray(xo), wi)
    for d in range(xi.shape[0]):
        ref = oracle.coalesce(*oracle.conservative_1d(xi[d], xo[d],
                                                      None if wi is None else wi[d]))
        for g, r in zip(got, ref):
            assert np.array_equal(g[off[d]:off[d + 1]], r, equal_nan=True), d


@pytest.mark.parametrize("reverse", [(1, 1), (-1, 1), (1, -1), (-1, -1)])
@pytest.mark.parametrize("n,m", [(2, 2), (2, 70), (1025, 3), (1026, 2048), (1024, 2049), (17, 16), (18, 31),
                                 (2100, 1500), (3, 2500), (4, 7000), (6000, 4000)])
def test_cells_match_oracle(n, m, reverse):
    rng = np.random.default_rng(n + m)
    xi = np.sort(rng.uniform(-1, 1, (3, n)), axis=1)
    xo = np.sort(rng.uniform(-1.2, 0.9, (3, m)), axis=1)
    k = min(n, m)
    xo[1, :k] = xi[1, :k]  # shared vertices
    xo[1] = np.sort(xo[1])
    _check(xi[:, :: reverse[0]], xo[:, :: reverse[1]], rng.uniform(0.5, 2, (3, n - 1)))


def test_unordered_elements_beside_ordered_ones():
    rng = np.random.default_rng(5)
    n, m = 1300, 1100
    xi = np.sort(rng.uniform(-1, 1, (9, n)), axis=1)
    xo = np.sort(rng.uniform(-1.2, 1.2, (9, m)), axis=1)
    xi[1, 700] = xi[1, 699]  # repeated
    xo[2, 300] = xo[2, 299]
    xi[3, [1100, 1200]] = xi[3, [1200, 1100]]  # unordered
    xo[4, [500, 600]] = xo[4, [600, 500]]
    xi[5, 1250] = np.nan
    xo[6, 40] = np.nan
    xi[7, 0], xo[7, -1] = -np.inf, np.inf
    with np.errstate(invalid="ignore"):
        _check(xi, xo)
