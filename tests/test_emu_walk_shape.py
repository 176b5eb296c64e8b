"""
The split of a build's sweeps into walk threads (``rg_walk_shape.hpp``, run on
the CPU through tests/emu): a coarse sweep does not make the others stage more,
alone or in a batch, and what a server reserves for a build covers its staging.
"""

import ctypes

import numpy as np
import pytest

from tests.emu import emu

MB = 1e6


def _shape(sizes):
    sizes = np.ascontiguousarray(sizes, dtype=np.int64).reshape(-1, 4)
    f = emu.lib().rge_walk_shape
    f.restype = ctypes.c_int64
    p = ctypes.POINTER(ctypes.c_int64)
    f.argtypes = [p, ctypes.c_int64, p]
    reserved = np.zeros(len(sizes), np.int64)
    return f(sizes.ctypes.data_as(p), len(sizes), reserved.ctypes.data_as(p)), reserved


def _edges(sizes):
    """Sweep edges, the rows of each pass padded to whole wavefronts."""
    t = 0
    for nxi, nyi, nxo, nyo in sizes:
        for a, b in ((nxi, nyi), (nyi, nxi), (nxo, nyo), (nyo, nxo)):
            t += (a + 63) // 64 * 64 * (b - 1)
    return t


# One-edge chunks stage at least 16 triples of 16 bytes; longer ones 1.8 times
# the expected triples (four to six an edge of grids of like spacing): 256
# bytes an edge at most where the coarse sweeps have few edges, as here.
@pytest.mark.parametrize("sizes", [
    [(9, 9, 400, 400)],
    [(400, 400, 9, 9)],
    [(200, 200, 150, 150), (9, 9, 300, 300)],
    [(33, 1025, 65, 2049)] + 20 * [(200, 210, 180, 170)],
    [(2049, 2049, 1537, 1537)],
    [(130, 70, 100, 100)],
])
def test_staging_of_uneven_pairs(sizes):
    staging, reserved = _shape(sizes)
    print(f"staging {staging / MB:.1f} MB, {staging / _edges(sizes):.0f} bytes an edge, "
          f"reserved {reserved.sum() / MB:.1f} MB")
    assert staging <= 256 * _edges(sizes) + 4 * MB
    assert reserved.sum() >= staging


@pytest.mark.parametrize("seed", range(20))
def test_reserved_bytes_cover_the_staging_of_batches(seed):
    r = np.random.default_rng(seed)
    for _ in range(50):
        n = int(r.integers(1, 40))
        sizes = np.exp(r.uniform(np.log(2), np.log(r.integers(3, 2000)), (n, 4))).astype(int)
        staging, reserved = _shape(np.maximum(sizes, 2))
        assert reserved.sum() >= staging
