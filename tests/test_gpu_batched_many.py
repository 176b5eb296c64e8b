"""
A batched apply of more blocks than one launch holds threads for (2^24 blocks
of 256): every image gets its result.
"""

import numpy as np
import pytest
import torch

from regridding_amd._lib import check, lib, rg_apply_job
from regridding_amd._regrid import import_weights

pytestmark = pytest.mark.gpu


def test_more_blocks_than_a_launch_holds():
    images = 8 * (2**24 + 5)  # eight to a block
    h = import_weights(np.array([0]), np.array([0]), np.array([3.0]), 1, 1)
    x = torch.arange(images, dtype=torch.float64, device="cuda")
    y = torch.full_like(x, -1)
    job = (rg_apply_job * 1)()
    job[0].weights, job[0].transpose, job[0].batch = h.ptr, 0, images
    job[0].values_input, job[0].values_output = x.data_ptr(), y.data_ptr()
    check(lib().rg_apply_batched_f64(job, 1, torch.cuda.current_stream().cuda_stream))
    assert int((y != 3 * x).sum()) == 0
