"""
The content digest of host arrays (``rg_digest_start`` / ``_finish``) on the
CPU, through the C entries alone.
"""

import ctypes

import numpy as np
import pytest

from regridding_amd._lib import LIB_PATH, load_library

L = load_library(LIB_PATH)


def _start(arrays):
    n = len(arrays)
    job = ctypes.c_void_p()
    st = L.rg_digest_start((ctypes.c_void_p * n)(*(a.ctypes.data for a in arrays)),
                           (ctypes.c_size_t * n)(*(a.nbytes for a in arrays)), n,
                           ctypes.byref(job))
    return st, job


def _digests(arrays):
    st, job = _start(arrays)
    assert st == 0
    out = (ctypes.c_uint64 * len(arrays))()
    assert L.rg_digest_finish(job, out) == 0
    return list(out)


def test_a_job_that_runs_out_of_memory_ends_with_an_error():
    # three arrays large enough for threads; the memory ends after the first
    arrays = [np.arange(200_000, dtype=np.float64) + k for k in range(3)]
    want = _digests(arrays)
    assert L.rg_inject_failure(b"digest") == 0
    st, job = _start(arrays)
    assert st != 0 and not job.value
    assert _digests(arrays) == want


@pytest.mark.parametrize("n", [40, 100_001])
def test_pairs_of_edits_show(n):
    """Two one-bit edits never cancel: in the same lane (eight words apart) or
    not, the first in any bit, the second in any bit, on several contents."""
    seen = 0
    for seed in range(2):
        a = np.random.default_rng(seed).normal(size=n)
        if seed:
            a[:] = 1.0
        ref, = _digests([a])
        bits = a.view(np.uint64)
        at = n // 2
        for apart in ((8, 1, 16) if n < 1000 else (8,)):
            first = range(64) if n < 1000 else (63, 62, 31, 0)
            for b0 in first:
                bits[at] ^= np.uint64(1 << b0)
                for b1 in range(64) if n < 1000 else range(0, 64, 6):
                    bits[at + apart] ^= np.uint64(1 << b1)
                    assert _digests([a]) != [ref], (seed, apart, b0, b1)
                    seen += 1
                    bits[at + apart] ^= np.uint64(1 << b1)
                bits[at] ^= np.uint64(1 << b0)
        assert _digests([a]) == [ref]
    assert seen > 50


def test_sign_and_small_change_show():
    v = np.random.default_rng(3).normal(size=1000)
    ref, = _digests([v])
    v[10] = -v[10]
    v[18:19].view(np.uint64)[0] ^= np.uint64(1 << 30)
    assert _digests([v]) != [ref]
