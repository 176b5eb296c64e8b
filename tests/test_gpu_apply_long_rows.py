"""
The apply without a plan on long rows, against a sequential sum, bit for bit:
a wavefront per row (64 entries on average, or 28 to 40 in few rows) and rows
of a wavefront that are long beside short ones, with lengths around the steps
the sums and chunks take, image counts around the passes, signed zeros,
infinities and NaN; alone, as jobs of one launch, and in a captured build and
apply.
"""

import numpy as np
import pytest
import torch

from oracle import oracle
from regridding_amd import _util, workloads
from regridding_amd._conservative import pack_pairs
from regridding_amd._lib import check, lib, rg_apply_job
from regridding_amd._regrid import import_weights
from regridding_amd.graph import BuildApplyGraph
from regridding_amd.torch_ops import regrid_apply

pytestmark = pytest.mark.gpu

N_IN = 900
STEPS = [15, 16, 17, 23, 24, 25, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256,
         257, 383, 384, 385, 400, 777]

# name: (row lengths, a wavefront per row)
LENGTHS = {
    "one": [800],
    "steps": STEPS + [0, 1, 7, 8, 9],
    "with_empty": [0, 300] * 20 + [0] * 3,
    "average_64": [64] * 130,
    "few_of_40": [40] * 90,
    "clumped": [0] * 30 + [500] * 20 + [0] * 500 + STEPS + [2] * 400,
    "average_39": [39] * 200,
}


def _weights(rng, lengths):
    col = [np.sort(rng.choice(N_IN, n, replace=False)) for n in lengths]
    i, j = np.concatenate(col), np.repeat(np.arange(len(lengths)), lengths)
    w = rng.normal(size=i.size)
    w[::7] = 0.0
    w[3::11] *= -1
    order = np.lexsort((j, i))
    return i[order], j[order], w[order]


def _sum(i, j, w, x, n_out):
    y = np.zeros((x.shape[0], n_out), x.dtype)
    with np.errstate(invalid="ignore"):
        for b in range(x.shape[0]):
            np.add.at(y[b], j, w.astype(x.dtype) * x[b, i])
    return y


def _values(rng, images, dtype):
    x = rng.normal(size=(images, N_IN)).astype(dtype)
    x[:, 5::50] = -0.0
    if images == 3:
        x[1, 7::300], x[1, 8::300], x[2, 9::300] = np.inf, -np.inf, np.nan
    return x


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("name", sorted(LENGTHS))
def test_long_rows(name, dtype):
    rng = np.random.default_rng(len(name))
    lengths = LENGTHS[name]
    i, j, w = _weights(rng, lengths)
    h = import_weights(i, j, w, N_IN, len(lengths))
    for images in (1, 2, 3, 5, 6, 8, 9):
        x = _values(rng, images, dtype)
        ref = _sum(i, j, w, x, len(lengths))
        got = regrid_apply(h, torch.from_numpy(x).cuda()).cpu().numpy()
        assert np.array_equal(got, ref, equal_nan=True), images
        assert np.array_equal(np.signbit(got[~np.isnan(got)]), np.signbit(ref[~np.isnan(ref)]))


def test_long_rows_as_jobs():
    rng = np.random.default_rng(5)
    made = [(name, images) for name in sorted(LENGTHS) for images in (1, 2, 8, 11)]
    handles, xs, refs = [], [], []
    for name, images in made:
        t = _weights(rng, LENGTHS[name])
        handles.append(import_weights(*t, N_IN, len(LENGTHS[name])))
        xs.append(_values(rng, images, np.float64))
        refs.append(_sum(*t, xs[-1], len(LENGTHS[name])))
    xs = [torch.from_numpy(x).cuda() for x in xs]
    ys = [torch.full(r.shape, np.nan, dtype=torch.float64, device="cuda") for r in refs]
    jobs = (rg_apply_job * len(made))()
    for job, h, x, y in zip(jobs, handles, xs, ys):
        job.weights, job.transpose, job.batch = h.ptr, 0, x.shape[0]
        job.values_input, job.values_output = x.data_ptr(), y.data_ptr()
    check(lib().rg_apply_batched_f64(jobs, len(made), torch.cuda.current_stream().cuda_stream))
    for m, y, r in zip(made, ys, refs):
        assert np.array_equal(y.cpu().numpy(), r, equal_nan=True), m


def test_long_rows_in_a_graph():
    pairs = []
    for si, so in (((101, 91), (4, 5)), ((60, 70), (55, 50)), ((33, 200), (3, 3))):
        ci, co, *_ = _util.normalize_coordinates(
            workloads.warped_grid(si, 0.3, 0.04, 0.03),
            workloads.warped_grid(so, 0.7, 0.0, 0.0, -0.9, 0.9), perturb=True, seed=11)
        pairs.append((ci, co))
    rng = np.random.default_rng(2)
    vals = [rng.normal(size=(b, (ci[0].shape[0] - 1) * (ci[0].shape[1] - 1)))
            for b, (ci, _) in zip((3, 2, 8), pairs)]
    g = BuildApplyGraph(pack_pairs(pairs), vals)
    try:
        for _ in range(2):
            g.launch()
            assert g.status() == 0
            for (ci, co), v, y in zip(pairs, vals, g.outputs()):
                n_out = (co[0].shape[0] - 1) * (co[0].shape[1] - 1)
                assert np.array_equal(y, oracle.apply(*oracle.weights_2d(ci, co), v, n_out))
    finally:
        g.close()
