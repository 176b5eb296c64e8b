"""
``rg_weights_set_shape`` between applies that stage input patches: the shape
only decides which rows and input cells share a patch, so every factorisation
of the cell counts gives the bits of the apply without a plan.
"""

import pytest
import torch

from regridding_amd import _util, workloads
from regridding_amd._conservative import build_2d
from regridding_amd._lib import check, lib
from regridding_amd.torch_ops import regrid_apply

pytestmark = pytest.mark.gpu

# cells of the grids, then other factorisations (the tiles' width and number
# stay the same from one to the next); at least 65536 outputs either way
SHAPES = [((330, 270), (300, 304)), ((330, 270), (304, 300)), ((270, 330), (304, 300)),
          ((297, 300), (300, 304)), ((330, 270), (300, 304))]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("transpose", [False, True])
def test_reshaped_weights_keep_their_results(transpose, dtype):
    (nxi, nyi), (nxo, nyo) = SHAPES[0]
    ci, co, *_ = _util.normalize_coordinates(
        workloads.warped_grid((nxi + 1, nyi + 1), 0.3, 0.03, 0.02),
        workloads.warped_grid((nxo + 1, nyo + 1), 0.05, 0.0, 0.0, -0.9, 0.9), perturb=True,
        seed=1)
    h = build_2d(ci, co)
    n = h.n_out if transpose else h.n_in
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn((4, n), dtype=dtype, device="cuda", generator=gen)
    check(lib().rg_set_apply_tuning(-16, 0, 0, -1))
    ref = regrid_apply(h, x, transpose=transpose)
    check(lib().rg_set_apply_tuning(16, 0, 0, -1))
    assert float(ref.abs().sum()) > 0
    for si, so in SHAPES:
        check(lib().rg_weights_set_shape(h.ptr, *si, *so))
        assert torch.equal(regrid_apply(h, x, transpose=transpose), ref), (si, so)
