"""
``rg_fill_gauss_seidel_2d`` on more slices than one launch holds threads for
(2^32, a workgroup of up to 512 for a slice): every slice of 2 x 2 cells gets
the result of the oracle's sweep of that slice.
"""

import numpy as np
import pytest
import torch

from oracle import oracle
from regridding_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def test_more_slices_than_a_launch_holds():
    T = 2**32 // 512 + 3
    r = np.random.default_rng(2)
    a = r.uniform(-1, 1, size=(1, 2, 2))
    where = np.array([[[True, False], [True, True]]])
    want = torch.as_tensor(oracle.fill_gauss_seidel_2d(a, where, 3), device="cuda")
    da = torch.as_tensor(a, device="cuda").expand(T, 2, 2).contiguous()
    dw = torch.as_tensor(where.astype(np.uint8), device="cuda").expand(T, 2, 2).contiguous()
    check(lib().rg_fill_gauss_seidel_2d(da.data_ptr(), dw.data_ptr(), T, 2, 2, 3,
                                        torch.cuda.current_stream().cuda_stream))
    assert int((da != want).any(2).any(1).sum()) == 0
