"""
The apply without a plan against a sequential sum, bit for bit: row lengths
around the chunks a wavefront takes, rows longer than a chunk, empty rows and
empty wavefronts, grid widths around 64, image counts around the split over
blocks, signed zeros, infinities and NaN; alone and as jobs of one launch.
"""

import numpy as np
import pytest
import torch

from regridding_amd._lib import check, lib, rg_apply_job
from regridding_amd._regrid import import_weights
from regridding_amd.torch_ops import regrid_apply

pytestmark = pytest.mark.gpu

N_IN = 700


def _weights(rng, lengths):
    """A CSR of these row lengths over N_IN columns, in storage order."""
    col = [np.sort(rng.choice(N_IN, n, replace=False)) for n in lengths]
    i = np.concatenate(col) if col else np.zeros(0, np.int64)
    j = np.repeat(np.arange(len(lengths)), lengths)
    w = rng.normal(size=i.size)
    w[::7] = 0.0
    w[3::11] *= -1
    order = np.lexsort((j, i))
    return i[order], j[order], w[order]


def _sum(i, j, w, x, n_out):
    """Rounded products added one at a time in order of the input cell."""
    y = np.zeros((x.shape[0], n_out), x.dtype)
    for b in range(x.shape[0]):
        np.add.at(y[b], j, w.astype(x.dtype) * x[b, i])
    return y


def _run_of(total, n=64):
    q, r = divmod(total, n)
    return [q + 1] * r + [q] * (n - r)


LENGTHS = {
    "empty": [0] * 130,
    "first": [1] + [0] * 200,
    "last": [0] * 191 + [5],
    "half": _run_of(191) + _run_of(192) + _run_of(193),
    "chunk": _run_of(383) + _run_of(384) + _run_of(385) + _run_of(10),
    "two": _run_of(575) + _run_of(576) + _run_of(577) + _run_of(769) + [2] * 7,
    "long": [3] * 20 + [700] + [0] * 5 + [650, 1, 384] + [2] * 90,
    "single": [9],
    "ragged": None,
}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("name", sorted(LENGTHS))
def test_row_lengths(name, dtype):
    rng = np.random.default_rng(len(name))
    lengths = LENGTHS[name]
    if lengths is None:
        lengths = rng.integers(0, 14, 1000) * (rng.random(1000) < 0.8)
    i, j, w = _weights(rng, lengths)
    n_out = len(lengths)
    h = import_weights(i, j, w, N_IN, n_out)
    for images in (1, 2, 3, 9):
        x = rng.normal(size=(images, N_IN)).astype(dtype)
        x[:, 5::50] = -0.0
        if images == 3:
            x[1, 7::90], x[1, 8::90], x[2, 9::90] = np.inf, -np.inf, np.nan
        with np.errstate(invalid="ignore"):
            ref = _sum(i, j, w, x, n_out)
        got = regrid_apply(h, torch.from_numpy(x).cuda()).cpu().numpy()
        assert np.array_equal(got, ref, equal_nan=True)
        assert np.array_equal(np.signbit(got[~np.isnan(got)]), np.signbit(ref[~np.isnan(ref)]))


@pytest.mark.parametrize("shape", [(5, 63), (5, 64), (7, 65), (3, 130), (9, 1), (1, 300), (2, 256)])
def test_grid_widths(shape):
    rng = np.random.default_rng(shape[1])
    n_out = shape[0] * shape[1]
    i, j, w = _weights(rng, rng.integers(0, 12, n_out))
    h = import_weights(i, j, w, N_IN, n_out)
    check(lib().rg_weights_set_shape(h.ptr, 20, 35, *shape))
    for images in (1, 4, 8):
        x = rng.normal(size=(images, N_IN))
        got = regrid_apply(h, torch.from_numpy(x).cuda()).cpu().numpy()
        assert np.array_equal(got, _sum(i, j, w, x, n_out))
    y = rng.normal(size=(2, n_out))
    back = regrid_apply(h, torch.from_numpy(y).cuda(), transpose=True).cpu().numpy()
    order = np.lexsort((i, j))
    assert np.array_equal(back, _sum(j[order], i[order], w[order], y, N_IN))


def test_jobs_match_alone():
    rng = np.random.default_rng(5)
    handles, xs = [], []
    for k, (images, shape) in enumerate([(1, (1, 1)), (8, (6, 65)), (9, (40, 10)), (17, (3, 200))]):
        n_out = shape[0] * shape[1]
        h = import_weights(*_weights(rng, rng.integers(0, 30, n_out)), N_IN, n_out)
        check(lib().rg_weights_set_shape(h.ptr, 20, 35, *shape))
        handles.append(h)
        xs.append(torch.from_numpy(rng.normal(size=(images, N_IN))).cuda())
    ys = [torch.full((x.shape[0], h.n_out), np.nan, dtype=x.dtype, device="cuda")
          for h, x in zip(handles, xs)]
    jobs = (rg_apply_job * len(handles))()
    for job, h, x, y in zip(jobs, handles, xs, ys):
        job.weights, job.transpose, job.batch = h.ptr, 0, x.shape[0]
        job.values_input, job.values_output = x.data_ptr(), y.data_ptr()
    check(lib().rg_apply_batched_f64(jobs, len(handles), torch.cuda.current_stream().cuda_stream))
    for h, x, y in zip(handles, xs, ys):
        assert torch.equal(y, regrid_apply(h, x))
