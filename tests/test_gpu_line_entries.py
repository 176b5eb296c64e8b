"""
The entries a block of 1-D conservative cells writes, around its windows of
2048: cells inside one output cell but one (entries = cells + breaks), with and
without a weighting, both directions, several elements side by side; the
oracle's triples, bit for bit.
"""

import numpy as np
import pytest

from tests.test_gpu_line_cells import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("reverse", [(1, 1), (-1, 1), (1, -1), (-1, -1)])
@pytest.mark.parametrize("cells,entries", [(1, 1), (1, 2047), (1, 2048), (1, 2049), (5, 4095),
                                           (5, 4096), (5, 4097), (1024, 2047), (1024, 2048),
                                           (1024, 2049), (1023, 6200), (1025, 2050)])
def test_windows(cells, entries, reverse, weighted):
    rng = np.random.default_rng(entries)
    xi = np.linspace(0, 1, cells + 1)[None] * np.array([[1.0], [1.5], [0.7]])
    # entries - cells output vertices inside, two outside
    breaks = np.sort(rng.uniform(0.001, 0.999, (3, entries - cells)), axis=1) * xi[:, -1:]
    xo = np.concatenate([np.full((3, 1), -0.5), breaks, np.full((3, 1), 2.0)], axis=1)
    assert (np.diff(xo, axis=1) > 0).all()
    wi = rng.uniform(0.5, 2, (3, cells)) if weighted else None
    _check(xi[:, :: reverse[0]], xo[:, :: reverse[1]], wi)
