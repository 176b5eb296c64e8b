"""
Weights edited so that they can no longer be used: the call raises, and a
caller's output buffer holds the zeros it was cleared to, nothing of the
weights as they were.
"""

import numpy as np
import pytest

import regridding_amd as rg
from regridding_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [20, 260])
def test_failing_import_leaves_the_buffer_cleared(n):
    gi = workloads.warped_grid(n, 0.2, 0.03, 0.04)
    go = workloads.warped_grid(n - 5, 0.45, 0.0, 0.0, -0.9, 0.9)
    w = rg.weights(gi, go, method="conservative")
    x = np.random.default_rng(1).normal(size=(3, n - 1, n - 1))
    out = np.full((3, n - 6, n - 6), np.nan)

    def apply():
        return rg.regrid_from_weights(*w, x, out, axis_input=(-2, -1), axis_output=(-2, -1))

    apply()
    assert np.abs(out).sum() > 0
    ii = w[0][()][0]
    good = ii[ii.size // 2]
    ii[ii.size // 2] = (n - 1) ** 2  # beyond the input cells
    with pytest.raises(Exception, match="out of range"):
        apply()
    assert np.array_equal(out, np.zeros_like(out))
    ii[ii.size // 2] = good
    y = apply()
    assert np.shares_memory(y, out)
    assert np.array_equal(y, rg.regrid_from_weights(*w, x, axis_input=(-2, -1),
                                                    axis_output=(-2, -1)))
