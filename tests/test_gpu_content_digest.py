"""
Weights edited in place are noticed whatever their size and wherever the edit
is: arrays hashed at once and in threads, lengths that are not whole blocks,
several host threads at a time; an output buffer of the caller's holds the
edited weights' result.
"""

import threading

import numpy as np
import pytest

import regridding_amd as rg
from oracle import oracle
from regridding_amd import _cache, workloads

pytestmark = pytest.mark.gpu


def _digest(a):
    return _cache._start_digest(a, a, a).result()


@pytest.mark.parametrize("n", [0, 1, 7, 8, 63, 64, 65, 128, 1000, 65535, 65536, 65537, 200001])
def test_every_change_shows(n):
    a = np.random.default_rng(n).normal(size=n)
    ref = _digest(a)
    assert _digest(a.copy()) == ref
    for q in {0, n // 3, n // 2, n - 1} if n else ():
        b = a.copy()
        b[q] = np.nextafter(b[q], 9)
        assert _digest(b) != ref
    assert _digest(np.append(a, 0.0)) != ref
    if n > 1:
        assert _digest(np.roll(a, 1)) != ref


@pytest.mark.parametrize("n", [20, 260])
@pytest.mark.parametrize("given", [False, True])
def test_edited_weights_are_applied(n, given):
    gi = workloads.warped_grid(n, 0.2, 0.03, 0.04)
    go = workloads.warped_grid(n - 5, 0.45, 0.0, 0.0, -0.9, 0.9)
    w = rg.weights(gi, go, method="conservative")
    ii, io, v = w[0][()]
    x = np.random.default_rng(1).normal(size=(3, n - 1, n - 1))
    out = np.full((3, n - 6, n - 6), np.nan) if given else None

    def apply():
        return rg.regrid_from_weights(*w, x, out, axis_input=(-2, -1), axis_output=(-2, -1))

    def ref():
        return oracle.apply(ii, io, v, x.reshape(3, -1), (n - 6) ** 2).reshape(3, n - 6, n - 6)

    assert np.array_equal(apply(), ref())
    v[v.size // 2] *= -3
    y = apply()
    assert np.array_equal(y, ref())
    assert not given or np.shares_memory(y, out)


def test_threads():
    pairs = [rg.weights(workloads.warped_grid(n, 0.2, 0.03, 0.04),
                        workloads.warped_grid(n + 9, 0.4, 0.0, 0.0, -0.9, 0.9),
                        method="conservative") for n in (30, 200, 230)]
    errors = []

    def work(k):
        try:
            for _ in range(5):
                w = pairs[k % 3]
                x = np.random.default_rng(k).normal(size=w[1])
                y = rg.regrid_from_weights(*w, x)
                ii, io, v = w[0][()]
                assert np.array_equal(y.ravel(), oracle.apply(ii, io, v, x.reshape(1, -1),
                                                              y.size)[0])
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
