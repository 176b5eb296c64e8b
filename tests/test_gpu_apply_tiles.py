"""
The staged apply in each tile width and kind of store its rule gives (rows of
whole cache lines or not, few or many images, more or fewer input than output
cells, short and long rows) against the apply without a plan, bit for bit.
"""

import numpy as np
import pytest
import torch

from regridding_amd import _util, workloads
from regridding_amd._conservative import build_2d
from regridding_amd._lib import check, lib
from regridding_amd.torch_ops import regrid_apply

pytestmark = pytest.mark.gpu

# (input, output) vertices and the image counts at either side of 130 MB
# (FP64) and 190 MB (FP32) of images
CASES = [((257, 257), (513, 257), (2, 9)),            # whole lines
         ((400, 331), (531, 487), (1, 2, 3, 8)),      # short rows, merged
         ((901, 890), (444, 460), (5, 17, 31)),       # long rows
         ((1100, 1013), (1201, 1180), (8, 9, 19)),    # near one to one
         ((720, 650), (1250, 1301), (10, 24)),        # rows of three; adjoint of nine
         ((1500, 1430), (1033, 1130), (6, 16))]


@pytest.fixture(autouse=True)
def _tuning():
    yield
    check(lib().rg_set_apply_tuning(16, 8, 32, 1))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0][0]}-{c[1][0]}")
def test_matches_unstaged(case, transpose, dtype):
    si, so, batches = case
    ci, co, *_ = _util.normalize_coordinates(
        workloads.warped_grid(si, 0.3, 0.03, 0.02),
        workloads.warped_grid(so, 0.05, 0.0, 0.0, -0.9, 0.9), perturb=True, seed=1)
    h = build_2d(ci, co)
    n = h.n_out if transpose else h.n_in
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn((max(batches), n), dtype=dtype, device="cuda", generator=gen)
    check(lib().rg_set_apply_tuning(-16, 0, 0, -1))
    ref = regrid_apply(h, x, transpose=transpose)
    check(lib().rg_set_apply_tuning(16, 0, 0, -1))
    assert float(ref.abs().sum()) > 0
    for b in batches:
        assert torch.equal(regrid_apply(h, x[:b], transpose=transpose), ref[:b])
