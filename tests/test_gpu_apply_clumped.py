"""
The apply without a plan where single wavefronts of 64 rows hold long rows: at
the number of entries from which such a wavefront takes its rows one after
another (more than 64 a row) and one either side, in full wavefronts and in
the last rows, spread evenly and in a few rows, against a sequential sum.
"""

import numpy as np
import pytest
import torch

from regridding_amd._lib import check, lib, rg_apply_job
from regridding_amd._regrid import import_weights

pytestmark = pytest.mark.gpu

N_IN = 900


def _lengths(total, last):
    even = [64] * 64
    even[17] += total - 64 * 64
    few = [0] * 64
    few[3:9] = [800, 1, 777, 0, 880, 64]
    few[40], few[63] = 700, total - 3222
    return [0] * 64 + even + [5] * 128 + few + [0] * 64 * 40 + last


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("total", [4095, 4096, 4097])
@pytest.mark.parametrize("last", [[200], [65, 64], [64, 64, 64], [0, 0, 193, 0], [97, 96]])
def test_clumped_rows(total, last, dtype):
    rng = np.random.default_rng(total + len(last))
    lengths = _lengths(total, last)
    col = [np.sort(rng.choice(N_IN, n, replace=False)) for n in lengths]
    i, j = np.concatenate(col), np.repeat(np.arange(len(lengths)), lengths)
    w = rng.normal(size=i.size)
    order = np.lexsort((j, i))
    i, j, w = i[order], j[order], w[order]
    h = import_weights(i, j, w, N_IN, len(lengths))
    made = [1, 2, 3, 5, 6, 8, 11]
    xs = [torch.from_numpy(rng.normal(size=(b, N_IN)).astype(dtype)).cuda() for b in made]
    ys = [torch.full((b, len(lengths)), np.nan, dtype=x.dtype, device="cuda")
          for b, x in zip(made, xs)]
    jobs = (rg_apply_job * len(made))()
    for job, x, y in zip(jobs, xs, ys):
        job.weights, job.transpose, job.batch = h.ptr, 0, x.shape[0]
        job.values_input, job.values_output = x.data_ptr(), y.data_ptr()
    run = lib().rg_apply_batched_f64 if dtype == np.float64 else lib().rg_apply_batched_f32
    check(run(jobs, len(made), torch.cuda.current_stream().cuda_stream))
    for x, y in zip(xs, ys):
        x, y = x.cpu().numpy(), y.cpu().numpy()
        ref = np.zeros_like(y)
        for b in range(x.shape[0]):
            np.add.at(ref[b], j, w.astype(dtype) * x[b, i])
        assert np.array_equal(y, ref), x.shape[0]
