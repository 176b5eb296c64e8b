"""
The staged apply on either side of each line its tile rule draws: output rows of
whole cache lines, of whole 64-byte pieces, and neither; images up to 50 MB, up
to 130 (FP64) or 190 MB (FP32), and beyond; fewer and more input than output
cells; weights of more and fewer than 4.5 (FP64) or 5.5 (FP32) a row.  Against
the apply without a plan, bit for bit.
"""

import numpy as np
import pytest
import torch

from regridding_amd import _util, workloads
from regridding_amd._conservative import build_2d
from regridding_amd._lib import check, lib
from regridding_amd.torch_ops import regrid_apply

pytestmark = pytest.mark.gpu

# (input, output) vertices; the cells of an output row make, in FP64 / FP32:
CASES = {
    "pieces_neither": ((451, 441), (401, 505)),   # 63 pieces / 31.5
    "lines_pieces": ((601, 513), (401, 529)),     # 33 lines / 33 pieces; adjoint 32 / 16 lines
    "neither": ((402, 431), (583, 632)),          # odd; few input cells
    "finer_in": ((700, 688), (462, 455)),         # odd; c = 2.3
    "near": ((520, 511), (488, 476)),             # c = 1.15
    "fine_out": ((330, 301), (650, 604)),         # c = 0.25; adjoint 4, rows of 300
}
LIMITS = {torch.float64: (50e6, 130e6), torch.float32: (50e6, 190e6)}


@pytest.fixture(autouse=True)
def _tuning():
    yield
    check(lib().rg_set_apply_tuning(16, 8, 32, 1))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("name", sorted(CASES))
def test_matches_unstaged(name, dtype):
    si, so = CASES[name]
    ci, co, *_ = _util.normalize_coordinates(
        workloads.warped_grid(si, 0.3, 0.03, 0.02),
        workloads.warped_grid(so, 0.05, 0.0, 0.0, -0.9, 0.9), perturb=True, seed=1)
    h = build_2d(ci, co)
    size = 8 if dtype == torch.float64 else 4
    per_image = (h.n_in + h.n_out) * size
    counts = [2]
    for limit in LIMITS[dtype]:  # on either side of it
        counts += [int(limit / per_image), int(limit / per_image) + 1]
    gen = torch.Generator(device="cuda").manual_seed(7)
    for transpose in (False, True):
        n = h.n_out if transpose else h.n_in
        x = torch.randn((max(counts), n), dtype=dtype, device="cuda", generator=gen)
        check(lib().rg_set_apply_tuning(-16, 0, 0, -1))
        ref = regrid_apply(h, x, transpose=transpose)
        check(lib().rg_set_apply_tuning(16, 0, 0, -1))
        assert float(ref.abs().sum()) > 0
        for b in counts:
            assert torch.equal(regrid_apply(h, x[:b], transpose=transpose), ref[:b]), b
