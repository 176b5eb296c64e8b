"""
The default split of the sweep into chunks (edges per walk thread by expected
work, one staging capacity for every pass) at the ends of its range: one edge
per chunk, the bound of a chunk, rows shorter than a chunk, sweeps so coarse
that an edge overflows the staging.  The result never depends on the split,
so every case equals the oracle bit for bit.
"""

import numpy as np
import pytest

from oracle import oracle
from regridding_amd import _util, workloads
from regridding_amd._conservative import build_2d, build_2d_batched

pytestmark = pytest.mark.gpu

PAIRS = {
    "smallest": ((2, 2), (2, 2)),
    "thin": ((3, 200), (150, 2)),
    "one_edge_overflows": ((3, 4), (301, 280)),
    "one_edge": ((67, 45), (39, 81)),
    "two_edges": ((300, 311), (290, 257)),
    "long_rows": ((9, 1500), (7, 1200)),
}


def _grids(name):
    si, so = PAIRS[name]
    gi = workloads.warped_grid(si, 0.3, 0.04, 0.03)
    go = workloads.warped_grid(so, 0.7, 0.0, 0.0, -0.9, 0.9)
    ci, co, *_ = _util.normalize_coordinates(gi, go, perturb=True, seed=11)
    return ci, co


def _same(got, exp):
    return all(np.array_equal(a, b) for a, b in zip(got, exp))


@pytest.mark.parametrize("name", sorted(PAIRS))
def test_default_chunks_match_oracle(name):
    ci, co = _grids(name)
    h = build_2d(ci, co)
    assert _same(h.export(), oracle.weights_2d(ci, co))
    if name == "one_edge_overflows":
        assert h.stats()["n_restaged"] > 0


def test_mixed_batch_matches_single_builds():
    pairs = [_grids(name) for name in sorted(PAIRS)]
    for h, (ci, co) in zip(build_2d_batched(pairs), pairs):
        assert _same(h.export(), oracle.weights_2d(ci, co))
    # the rule's chunks against the same 16 edges for every pass
    for h, g in zip(build_2d_batched(pairs), build_2d_batched(pairs, edges_per_lane=16)):
        assert _same(h.export(), g.export())
