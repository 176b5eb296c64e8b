"""
Device residency of weights returned to the host.

``weights()`` must return host arrays (the reference's flat
``(indices_input, indices_output, values)`` triples,
``regridding/_weights/_weights.py:31-36``), but the device already holds
them as CSR after the build.  This registry remembers, for each returned
triple, the device handle it came from, so ``regrid_from_weights`` on those
very arrays (or on their ``transpose_weights`` swap) applies the resident
CSR instead of uploading and regrouping the triples again.

Entries are keyed by the identity of the three arrays and die with them.
A triple may also be registered as part ``d`` of ``D`` of a block-diagonal
handle (the 1-D builders put all elements of one call in one handle).
The arrays stay writable, as the reference returns them
(``_weights_arrays.py:68-72``): each entry records a digest of the
three arrays' bytes, and a hit counts only while the arrays still hash to
it, so a caller who edits the weights in place gets the edited weights
applied (one pass over the arrays per lookup, in native threads;
``lookup_pending`` lets it run beside the copies of the values).
Arrays the registry has not seen (unpickled, hand-made, modified) go
through the import path.
"""

from __future__ import annotations

import ctypes
import threading
import weakref

import numpy as np

from ._lib import Weights, check, lib

__all__ = ["register", "lookup"]

_lock = threading.Lock()
# id(values) -> (weakref(indices_input), weakref(indices_output), Weights, part, digest)
_entries: dict[int, tuple] = {}


def _drop(key: int) -> None:
    with _lock:
        _entries.pop(key, None)


class _Digest:
    """A content digest of a triple in the making (input and output roles told
    apart by their order)."""

    def __init__(self, arrays: tuple[np.ndarray, ...]):
        self._job = None
        self._arrays = arrays
        n = len(arrays)
        job = ctypes.c_void_p()
        check(lib().rg_digest_start((ctypes.c_void_p * n)(*(x.ctypes.data for x in arrays)),
                                    (ctypes.c_size_t * n)(*(x.nbytes for x in arrays)), n,
                                    ctypes.byref(job)))
        self._job = job.value

    def result(self) -> tuple:
        """The digest; once only."""
        job, self._job = self._job, None
        out = (ctypes.c_uint64 * len(self._arrays))()
        check(lib().rg_digest_finish(job, out))
        return tuple((x.dtype.str, x.shape, h) for x, h in zip(self._arrays, out))

    def __del__(self):
        if self._job is not None:  # the threads read the arrays
            self.result()


def _start_digest(a: np.ndarray, b: np.ndarray, values: np.ndarray) -> _Digest | None:
    """None when an array is not C-contiguous or holds objects."""
    arrays = (a, b, values)
    if any(not x.flags.c_contiguous or x.dtype.hasobject for x in arrays):
        return None
    return _Digest(arrays)


def register(indices_input: np.ndarray, indices_output: np.ndarray, values: np.ndarray,
             handle: Weights, part: tuple[int, int, int, int] | None = None) -> None:
    """``part``: ``(d, D, n_in, n_out)`` when ``handle`` is block-diagonal
    and this triple is its block d (n_in x n_out cells per block)."""
    digest = _start_digest(indices_input, indices_output, values)
    if digest is None:
        return
    digest = digest.result()
    key = id(values)
    with _lock:
        _entries[key] = (weakref.ref(indices_input), weakref.ref(indices_output), handle, part,
                         digest)
    weakref.finalize(values, _drop, key)


def lookup(a: np.ndarray, b: np.ndarray, values: np.ndarray) -> tuple[Weights, bool] | None:
    """
    ``(handle, transposed)`` if ``(a, b, values)`` is a registered whole
    triple (``transposed=False``) or its index swap (``transposed=True``).
    """
    hit = lookup_part(a, b, values)
    if hit is None or hit[2] is not None:
        return None
    return hit[0], hit[1]


def lookup_part(a: np.ndarray, b: np.ndarray, values: np.ndarray):
    """``(handle, transposed, part)`` for a registered triple or its swap
    (``part`` None for a whole handle), else None."""
    hit = _find(a, b, values)
    if hit is None or not _Pending(*hit).unchanged():
        return None
    return hit[1:4]


def lookup_block(a: np.ndarray, b: np.ndarray, values: np.ndarray):
    """:func:`lookup_part` where only a block of a block-diagonal handle
    counts; the arrays of a whole handle are not read."""
    hit = _find(a, b, values)
    if hit is None or hit[3] is None or not _Pending(*hit).unchanged():
        return None
    return hit[1:4]


def lookup_pending(a: np.ndarray, b: np.ndarray, values: np.ndarray):
    """``(handle, transposed, pending)`` like :func:`lookup`, but the arrays
    are still being compared with what was registered: what is computed from
    the handle holds only if ``pending.unchanged()``."""
    hit = _find(a, b, values)
    if hit is None or hit[3] is not None:
        return None
    return hit[1], hit[2], _Pending(*hit)


class _Pending:
    def __init__(self, arrays, handle, transposed, part, digest):
        self._key, self._expected = id(arrays[2]), digest
        self._digest = _start_digest(*arrays)

    def unchanged(self) -> bool:
        """Whether the arrays still are what was registered (asked once); an
        entry whose arrays have changed is dropped."""
        if self._digest is not None and self._digest.result() == self._expected:
            return True
        _drop(self._key)
        return False


def _find(a: np.ndarray, b: np.ndarray, values: np.ndarray):
    """The entry of these arrays, their content not looked at:
    ``((indices_input, indices_output, values), handle, transposed, part,
    digest)``."""
    with _lock:
        e = _entries.get(id(values))
    if e is None:
        return None
    ri, ro, handle, part, digest = e
    ii, io = ri(), ro()
    if ii is None or io is None:
        return None
    if a is ii and b is io:
        transposed = False
    elif a is io and b is ii:
        transposed = True
    else:
        return None
    return (ii, io, values), handle, transposed, part, digest
