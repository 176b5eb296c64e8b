"""
The group reduction with output cells counted from the group's smallest (as
builds of hundreds of millions of triples do), forced to 13 bits: groups whose
outputs fit, groups too widely spread, which take the general reduction, and
both in one build, alone and in a batch, against the oracle, bit for bit.
"""

import numpy as np
import pytest

from oracle import oracle
from regridding_amd import _util, workloads
from regridding_amd._conservative import build_2d, build_2d_batched

pytestmark = pytest.mark.gpu

REDUCE_NEAR = 16  # RG_TUNE_REDUCE_NEAR

# name: (input shape, output shape, rotation of the output)
GRIDS = {
    "fit": ((120, 131), (75, 80), 0.1),
    "rows_of_64": ((90, 66), (140, 60), 0.02),
    "both": ((70, 80), (100, 130), 1.3),
    "spread": ((60, 65), (200, 210), 0.9),
    "coarse_in": ((20, 18), (130, 150), 0.6),
    "sparse": ((150, 141), (40, 37), 0.2),
}


def _grids(name):
    si, so, theta = GRIDS[name]
    gi = workloads.warped_grid(si, 0.05, 0.03, 0.03)
    go = workloads.warped_grid(so, theta, 0.0, 0.0, -0.9, 0.9)
    ci, co, *_ = _util.normalize_coordinates(gi, go, perturb=True, seed=3)
    return ci, co


def _spread(ci, co):
    """Largest minus smallest output cell of each group of 64 input cells."""
    i, o, _ = oracle.sweep_2d(ci, co)
    g = np.asarray(i) // 64
    lo = np.full(g.max() + 1, np.iinfo(np.int64).max)
    hi = np.full(g.max() + 1, -1)
    np.minimum.at(lo, g, o)
    np.maximum.at(hi, g, o)
    return (hi - lo)[hi >= 0]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("name", sorted(GRIDS))
def test_groups_match_oracle(name, weighted):
    ci, co = _grids(name)
    wi = None
    if weighted:
        wi = np.random.default_rng(4).uniform(0.5, 2, tuple(s - 1 for s in ci[0].shape))
    got = build_2d(ci, co, wi, flags=REDUCE_NEAR).export()
    for a, b in zip(got, oracle.weights_2d(ci, co, wi)):
        assert np.array_equal(a, b)


def test_batch_matches_oracle():
    pairs = [_grids(n) for n in sorted(GRIDS)]
    for h, (ci, co) in zip(build_2d_batched(pairs, flags=REDUCE_NEAR), pairs):
        for a, b in zip(h.export(), oracle.weights_2d(ci, co)):
            assert np.array_equal(a, b)


def test_grids_cover_both():
    s = {n: _spread(*_grids(n)) for n in GRIDS}
    assert (s["fit"] < 8192).all() and (s["spread"] >= 8192).any()
    assert (s["both"] < 8192).any() and (s["both"] >= 8192).any()
