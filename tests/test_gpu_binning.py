"""assign_to_cell's order within cells: the list build windows each run of cells by x, so a cell out
of order loses pairs.  Cell sizes around the edges of the ranking (a half wavefront, a wavefront,
several), with many molecules at equal x, against the oracle's cells and neighbour set."""
import sys

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd.md import MDContext
from oracle.oracle import Oracle
from tests.helpers import canonical_pairs

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def cell_filled(counts, seed):
    """Molecules in a box of 5^3 cells of side 2.8: counts[c] in cell c (x fastest), x from six
    values a cell (one of them for both of two molecules in three), y and z uniform."""
    rng = np.random.default_rng(seed)
    r = []
    for c, k in enumerate(counts):
        lo = 2.8 * np.array([c % 5, (c // 5) % 5, c // 25]) - 7.0
        q = rng.uniform(0.01, 2.79, (k, 3))
        q[:, 0] = np.linspace(0.1, 2.7, 6)[rng.integers(0, 6, k)]
        r.append(lo + q)
    return np.concatenate(r)


@pytest.mark.parametrize("counts", [
    (0, 1, 2, 31, 32, 33, 63, 64, 65, 128, 129, 200),   # mean below 24: two cells a wavefront
    (25, 26, 31, 32, 33, 40, 63, 64, 65, 70),           # mean above 24: one cell a wavefront
])
def test_cells_of_any_size(counts):
    n = np.array([counts[c % len(counts)] if len(counts) == 10 or c < 24 else 3 for c in range(125)])
    r = cell_filled(n, seed=31)
    r = r[np.random.default_rng(5).permutation(r.shape[0])]
    p = config.make_params((14.0, 14.0, 14.0), r.shape[0] / 14.0 ** 3, 2.5, tplot=10)
    p.brick[0] = p.brick[1] = p.brick[2] = 1
    say(f"case: {r.shape[0]} molecules, cells of {sorted(set(counts))}")
    o, g = Oracle(p, r, np.zeros_like(r)), MDContext(p, r, np.zeros_like(r))
    for x in (o, g):
        x.assign_to_cell()
    assert np.array_equal(g.cells(), o.cells())
    o.updateborders(1)
    o.assign_to_neighbourlist()
    g.messenger_updateborders(1)
    g.assign_to_neighbourlist()
    assert np.array_equal(canonical_pairs(*o.neighbourlist()), canonical_pairs(*g.neighbourlist()))
    g.close()
