"""
``regrid_apply`` recorded in a graph after an eager apply of another image
count, whose plan has another tile width or which made none: every replay
gives the eager result.
"""

import pytest
import torch

from regridding_amd import _util, workloads
from regridding_amd._conservative import build_2d
from regridding_amd.torch_ops import regrid_apply

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grids():
    ci, co, *_ = _util.normalize_coordinates(
        workloads.warped_grid((640, 650), 0.3, 0.03, 0.02),
        workloads.warped_grid((701, 690), 0.05, 0.0, 0.0, -0.9, 0.9), perturb=True, seed=1)
    return ci, co


# images of the eager calls before, and of the captured call.  FP64: up to 130
# MB of images (17 here) one width, beyond it another; FP32: up to 190 MB (49).
@pytest.mark.parametrize("before,images", [((1,), 4), ((4,), 24), ((24,), 3), ((3, 60), 4),
                                           ((1,), 60), ((60,), 5)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("transpose", [False, True])
def test_captured_after_other_image_counts(grids, before, images, dtype, transpose):
    h = build_2d(*grids)
    n = h.n_out if transpose else h.n_in
    for b in before:
        regrid_apply(h, torch.rand((b, n), dtype=dtype, device="cuda"), transpose=transpose)
    x = torch.rand((images, n), dtype=dtype, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = regrid_apply(h, x, transpose=transpose)
    for k in range(3):
        x.copy_(torch.rand(x.shape, dtype=dtype, device="cuda"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, regrid_apply(h, x, transpose=transpose)), k
