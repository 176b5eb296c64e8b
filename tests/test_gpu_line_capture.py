"""
``rg_conservative_1d_emit`` recorded in a graph (it takes no memory of its
own there): every replay, with other eager calls in between, gives the triples
of the eager call, for ordered elements and for those that need the serial
sweep.
"""

import ctypes

import numpy as np
import pytest
import torch

from regridding_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1300, 900), (40, 2500), (9, 7)])
def test_captured_emit(n, m):
    D, L = 37, lib()
    rng = np.random.default_rng(n)
    xi = np.sort(rng.uniform(-1, 1, (D, n)), axis=1)
    xo = np.sort(rng.uniform(-1.2, 1.2, (D, m)), axis=1)
    xi[3, 5] = xi[3, 4]  # repeated, unordered, NaN
    xi[7, [2, 6]] = xi[7, [6, 2]]
    xo[11, [1, 5]] = xo[11, [5, 1]]
    xo[12, 3] = np.nan
    xi[20:] = xi[20:, ::-1]
    xo[30:] = xo[30:, ::-1]
    s = lambda: torch.cuda.current_stream().cuda_stream  # noqa: E731
    x, o, wi = (torch.as_tensor(np.ascontiguousarray(v), device="cuda")
                for v in (xi, xo, rng.uniform(0.5, 2, (D, n - 1))))
    counts = torch.empty(D * (n - 1), dtype=torch.int32, device="cuda")
    offsets = torch.empty(D * (n - 1) + 1, dtype=torch.int64, device="cuda")
    total = ctypes.c_int64()
    check(L.rg_conservative_1d_count(x.data_ptr(), n, o.data_ptr(), m, D, counts.data_ptr(),
                                     offsets.data_ptr(), ctypes.byref(total), s()))
    T = total.value
    assert T > 0

    def emit(out):
        check(L.rg_conservative_1d_emit(x.data_ptr(), n, o.data_ptr(), m, D, wi.data_ptr(),
                                        counts.data_ptr(), offsets.data_ptr(),
                                        *(v.data_ptr() for v in out), s()))

    types = (torch.int64, torch.int64, torch.float64)
    want = [torch.empty(T, dtype=t, device="cuda") for t in types]
    emit(want)
    got = [torch.empty(T, dtype=t, device="cuda") for t in types]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        emit(got)
    for _ in range(3):
        for v in got:
            v.fill_(-7)
        g.replay()
        for v, w in zip(got, want):
            assert torch.equal(v.view(torch.int64), w.view(torch.int64))
        emit([torch.empty_like(w) for w in want])
        torch.cuda.synchronize()
