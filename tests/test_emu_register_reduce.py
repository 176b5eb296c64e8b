"""The register reduction of the build (keys as doubles, their sorting network
and the runs' sums: KeyBits, sort_doubles, run_heads and sum_runs, shared by the
GPU kernels and the CPU emulation) against a stable sort and np.add.reduceat:
every size of network, cells from empty to full, the widest keys, output cells
counted from the group's smallest, and runs at the longest sequential sum."""

import numpy as np
import pytest

from tests.emu import emu

SIZES = [8, 16, 24, 32, 48, 64]


def _cell(rng, n, triples, outs):
    ordinal = rng.choice(min(triples, 10**6), n, replace=False) + max(0, triples - 10**6)
    out = rng.choice(outs, n)
    vals = rng.normal(size=n) * 10.0 ** rng.integers(-8, 8, size=n)
    vals[rng.random(n) < 0.1] = -0.0
    return (out.astype(np.uint64) << np.uint64(32)) | ordinal.astype(np.uint64), vals


def _check(m, triples, most_out, keys, vals, out0=0):
    c, near, po, pv = emu.registers_reduce(m, triples, most_out, keys, vals, out0)
    order = np.argsort(keys, kind="stable")
    out = (keys[order] >> np.uint64(32)).astype(np.int64)
    starts = np.flatnonzero(np.r_[True, out[1:] != out[:-1]]) if len(out) else np.zeros(0, int)
    longest = max(np.diff(np.r_[starts, len(out)]), default=0)
    if longest > 8:
        assert c == -1
        return near
    assert c == len(starts)
    assert np.array_equal(po.astype(np.int64) + (out0 if near else 0), out[starts])
    if c:
        ref = np.add.reduceat(vals[order], starts)
        assert np.array_equal(pv, ref) and np.array_equal(np.signbit(pv), np.signbit(ref))
    return near


@pytest.mark.parametrize("m", SIZES)
def test_cells_of_every_size(m):
    rng = np.random.default_rng(m)
    for n in range(m + 1):
        for few in (1, 3, 8, 40):
            triples, most_out = 50_000_000, 2_400_000
            outs = rng.choice(most_out, few, replace=False)
            outs[0] = most_out - 1
            assert not _check(m, triples, most_out, *_cell(rng, n, triples, outs))


@pytest.mark.parametrize("m", SIZES)
def test_every_zero_one_key_sorts(m):
    # (by the 0-1 principle; all of them for 8, random ones for the others)
    rng = np.random.default_rng(m)
    rows = ([[r >> b & 1 for b in range(8)] for r in range(256)] if m == 8
            else rng.integers(0, 2, (300, m)))
    for row in rows:
        # the ordinals keep the records' order, so each run is its values in turn
        keys = (np.array(row, np.uint64) << np.uint64(32)) | np.arange(m, dtype=np.uint64)
        _check(m, 1000, 2, keys, rng.normal(size=m))


@pytest.mark.parametrize("triples,most_out,near", [
    (2**32 - 1, 2**23, False), (2**32 - 1, 2**23 + 1, True), (2**32 - 1, 2**31 - 1, True),
    (719_000_000, 33_640_000, True), (2, 2**31 - 1, False), (1, 1, False),
    (2**24, 2**31 - 1, False), (2**24 + 1, 2**31 - 1, True)])
def test_widest_keys(triples, most_out, near):
    rng = np.random.default_rng(most_out % 1000)
    for m in SIZES:
        for out0 in (0, max(0, most_out - 5000)):
            n = min(m, triples)
            span = min(most_out - out0, 2**23 if near else most_out)
            outs = out0 + rng.integers(0, span, 20)
            outs[:2] = out0, out0 + span - 1
            keys, vals = _cell(rng, n, triples, outs)
            assert _check(m, triples, most_out, keys, vals, out0) == near
