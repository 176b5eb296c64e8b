"""
A replay that outgrows only the graph's overflow buffer (its triples in all
fit): chunks past the buffer's end keep nothing, so records of the buckets
stay unwritten, and the reduction keeps nothing of that replay.  The graph
says so, and the next replay that fits is right again.
"""

import numpy as np
import pytest

from oracle import oracle
from regridding_amd import _util, workloads
from regridding_amd._conservative import pack_pairs
from regridding_amd._lib import RGError
from regridding_amd.graph import BuildApplyGraph

pytestmark = pytest.mark.gpu

OVERFLOW = 2


def _pair(power, seed):
    """Input vertices crowded around the middle for a power above 1: as many
    crossings in all, most of them in few chunks."""
    x, y = workloads.warped_grid((121, 111), 0.0, 0.0, 0.0, -1.0, 1.0)
    crowd = lambda v: np.sign(v) * np.abs(v) ** power  # noqa: E731
    ci, co, *_ = _util.normalize_coordinates(
        (crowd(x), crowd(y)), workloads.warped_grid((97, 83), 0.4, 0.0, 0.0, -0.6, 0.6),
        perturb=True, seed=seed)
    return ci, co


def test_overflow_alone_is_flagged_and_left():
    even = [_pair(1.0, 42) for _ in range(3)]
    crowded = [_pair(9.0, 42) for _ in range(3)]
    packed = pack_pairs(even)
    vals = [np.random.default_rng(k).normal(size=(2, 120 * 110)) for k in range(3)]
    g = BuildApplyGraph(packed, vals, slack=3.0, edges_per_lane=16, stage_per_edge=8)
    try:
        g.launch()
        assert g.status() == 0
        want = [o.copy() for o in g.outputs()]
        for _ in range(2):
            packed.update(crowded)
            g.launch()
            f = g.status()
            print(f"capacity {g.capacity()}, status {f:#x}", flush=True)
            assert f & OVERFLOW and not f & 1
            with pytest.raises(RGError):
                g.weights(0)
            for o, w in zip(g.outputs(), want):  # no apply of it ran
                assert np.array_equal(o, w)
            packed.update(even)
            g.launch()
            assert g.status() == 0
            for k, o in enumerate(g.outputs()):
                ii, io, w = oracle.weights_2d(*even[k])
                for a, b in zip(g.weights(k).export(), (ii, io, w)):
                    assert np.array_equal(a, b)
                assert np.array_equal(o, want[k])
    finally:
        g.close()
