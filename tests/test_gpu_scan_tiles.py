"""
The device-wide scans at the edges of their tiles (2048 items) and of the scan
of the tile sums (1024 tiles): the offsets of 1-D conservative weights are the
running sums of their counts.
"""

import ctypes

import numpy as np
import pytest
import torch

from regridding_amd._lib import check, lib

pytestmark = pytest.mark.gpu

TILE, SELF = 2048, 1024


@pytest.mark.parametrize("cells", [1, 2, 255, 256, 257, TILE - 1, TILE, TILE + 1, 3 * TILE + 7,
                                   SELF * TILE - 1, SELF * TILE, SELF * TILE + 1,
                                   (SELF + 5) * TILE + 1000])
def test_offsets_are_running_sums(cells):
    n, m = cells + 1, 2 * cells // 3 + 2
    x = torch.linspace(0, 1, n, dtype=torch.float64, device="cuda")
    y = torch.linspace(0.05, 0.95, m, dtype=torch.float64, device="cuda")
    counts = torch.empty(cells, dtype=torch.int32, device="cuda")
    offsets = torch.full((cells + 1,), -1, dtype=torch.int64, device="cuda")
    total = ctypes.c_int64()
    check(lib().rg_conservative_1d_count(x.data_ptr(), n, y.data_ptr(), m, 1, counts.data_ptr(),
                                         offsets.data_ptr(), ctypes.byref(total),
                                         torch.cuda.current_stream().cuda_stream))
    ref = np.concatenate([[0], np.cumsum(counts.cpu().numpy(), dtype=np.int64)])
    assert np.array_equal(offsets.cpu().numpy(), ref)
    assert total.value == ref[-1] and ref[-1] > 0
