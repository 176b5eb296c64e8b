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
