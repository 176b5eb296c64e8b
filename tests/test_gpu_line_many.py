"""
The 1-D conservative passes on more elements than one launch holds blocks of
256 threads for (2^24): every element gets the same triples as the first, and
the first those of the oracle.
"""

import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle
from regridding_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def test_more_elements_than_a_launch_holds():
    D, n, m = 2**24 + 3, 48, 2
    xi = np.linspace(0, 1, n)
    xo = xi[[20, 21]] + 0.3 / n  # a cell over two input cells
    want = oracle.coalesce(*oracle.conservative_1d(xi, xo, None))
    s = torch.cuda.current_stream().cuda_stream
    x, o = (torch.as_tensor(v, device="cuda").expand(D, v.size).contiguous() for v in (xi, xo))
    counts = torch.empty(D * (n - 1), dtype=torch.int32, device="cuda")
    offsets = torch.empty(D * (n - 1) + 1, dtype=torch.int64, device="cuda")
    total = ctypes.c_int64()
    check(lib().rg_conservative_1d_count(x.data_ptr(), n, o.data_ptr(), m, D, counts.data_ptr(),
                                         offsets.data_ptr(), ctypes.byref(total), s))
    assert total.value == D * want[0].size
    got = [torch.full((total.value,), -7, dtype=t, device="cuda")
           for t in (torch.int64, torch.int64, torch.float64)]
    check(lib().rg_conservative_1d_emit(x.data_ptr(), n, o.data_ptr(), m, D, None,
                                        counts.data_ptr(), offsets.data_ptr(),
                                        *(g.data_ptr() for g in got), s))
    for g, r in zip(got, want):
        assert int((g.reshape(D, -1) != torch.as_tensor(r, device="cuda")).sum()) == 0
