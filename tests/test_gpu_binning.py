"""assign_to_cell's order within cells: the list build windows each run of cells by x, so a cell out
of order loses pairs.  Cell sizes around the edges of the ranking (a half wavefront, a wavefront,
several), with many molecules at equal x, against the oracle's cells and neighbour set."""
import sys

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd._abi import FM_ENSEMBLE_TAG_MOVE, FM_INTEGRATION_LFV, FM_TAG_FIXED_SLIDE
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


def near_faces(r, L, count, corners, lo, hi, seed):
    """r with `count` molecules moved to between lo and hi beyond an upper face of the box (a lower one
    too when lo is positive), `corners` of them at two or three faces."""
    rng = np.random.default_rng(seed)
    r = r.copy()
    for k, n in enumerate(rng.permutation(r.shape[0])[:count]):
        for ax in rng.permutation(3)[: (2 + k % 2) if k < corners else 1]:
            side = rng.choice([-1.0, 1.0]) if lo >= 0.0 else 1.0
            r[n, ax] = side * (0.5 * L[ax] + rng.uniform(lo, hi))
    return r


@pytest.mark.parametrize("count,corners", [(0, 0), (1, 0), (63, 0), (65, 1), (1024, 0), (1025, 0), (1025, 3),
                                           (2048, 0), (2049, 0), (2500, 40)])
def test_renumbering_of_any_leaver_count(count, corners):
    """sendmols' numbers and positions, alone and inside the binning of a queued rebuild, for leaver
    counts around the wavefront, the workgroup and its LDS, with and without molecules that leave
    across an edge."""
    say(f"case: {count} of 3960 molecules outside the box, {corners} across edges")
    p, r, v = config.config_fcc((10, 9, 11), 0.8, 2.5, seed=8, tplot=1)
    out = near_faces(r, p.domain, count, corners, 0.0, 0.3, seed=9)
    o, g = Oracle(p, out, v), MDContext(p, out, v)
    for x in (o, g):
        x.sendmols()
    for ref, got in zip(o.state()[:2], g.state()[:2]):
        assert np.array_equal(ref, got)
    g.close()
    # the queued rebuild: every molecule slides by 0.2 along x, y and z a step, whatever its force
    p.ensemble, p.integration_algorithm = FM_ENSEMBLE_TAG_MOVE, FM_INTEGRATION_LFV
    for d in range(3):
        p.wallslidev[d] = 0.2 / p.delta_t
    inside = near_faces(r, p.domain, count, corners, -0.19, -0.01, seed=9)
    ends = []
    for queued in (False, True):
        g = MDContext(p, inside, v)
        g.set_tags(np.full(r.shape[0], FM_TAG_FIXED_SLIDE, np.int32))
        g.setup(0)
        if queued:
            g.run_lfv(0, 3)
        else:
            for it in range(3):
                g.md_advance_lfv(it)
        ends.append(g.state() + (g.rtether(),))
        g.close()
    for ref, got in zip(*ends):
        assert np.array_equal(ref, got, equal_nan=True)


def sparse(cells, seed):
    """A box of cells^3 cells of side 2.8, nearly all empty: clumps of up to 130 molecules in cells here
    and there, with many at equal x, and single molecules."""
    rng = np.random.default_rng(seed)
    r = []
    for k in [1, 2, 3, 5, 31, 32, 33, 63, 64, 65, 130] * 12 + [1] * 2000:
        q = rng.uniform(0.01, 2.79, (k, 3))
        if k > 3:
            q[:, 0] = np.linspace(0.1, 2.7, 6)[rng.integers(0, 6, k)]
        r.append(2.8 * (rng.integers(0, cells, 3) - 0.5 * cells) + q)
    r = np.concatenate(r)
    return r[rng.permutation(r.shape[0])]


@pytest.mark.parametrize("cells", [26, 66])      # the scan of the counts by itself, and from the chunks' sums
def test_cells_of_few_molecules(cells):
    r = sparse(cells, seed=cells)
    L = 2.8 * cells + 1e-9
    p = config.make_params((L, L, L), r.shape[0] / L ** 3, 2.5, tplot=10, ensemble=FM_ENSEMBLE_TAG_MOVE)
    p.brick[0] = p.brick[1] = p.brick[2] = 3
    say(f"case: {r.shape[0]} molecules in {cells}^3 cells")
    rng = np.random.default_rng(1)
    tag = rng.choice(np.array([0, FM_TAG_FIXED_SLIDE], np.int32), r.shape[0])
    o, g = Oracle(p, r, np.zeros_like(r)), MDContext(p, r, np.zeros_like(r))
    g.set_tags(tag, r + 1.0)
    for x in (o, g):
        x.assign_to_cell()
    assert np.array_equal(g.cells(), o.cells())
    for got, ref in zip(g.state()[:2] + (g.labels()[0], g.rtether()), (r, np.zeros_like(r), tag, r + 1.0)):
        assert np.array_equal(got, ref)
    o.updateborders(1)
    o.assign_to_neighbourlist()
    g.messenger_updateborders(1)
    g.assign_to_neighbourlist()
    assert np.array_equal(canonical_pairs(*o.neighbourlist()), canonical_pairs(*g.neighbourlist()))
    for _ in range(2):                            # the counts are ready for the next binning
        g.assign_to_cell()
        assert np.array_equal(g.cells(), o.cells())
    g.close()


def test_gas_loop_equals_the_routines():
    """A gas of two molecules a cell, rebuilt every third step: the fused loop's rebuilds (leavers wrapped and
    counted in one launch) against the routines', bit for bit."""
    say("case: 32000 molecules at density 0.1, 30 steps")
    p, r, v = config.config_fcc((20, 20, 20), 0.08, 2.5, seed=4, tplot=3)
    r = r + np.random.default_rng(2).uniform(-0.2, 0.2, r.shape)
    L = np.array([p.domain[d] for d in range(3)])
    r = np.where(r < -0.5 * L, r + L, np.where(r >= 0.5 * L, r - L, r))
    a, b = MDContext(p, r, 3.0 * v), MDContext(p, r, 3.0 * v)
    assert np.prod(a.geometry()["ncells"]) >= 16384
    a.setup(0)
    b.setup(0)
    a.run_vv(1, 30)
    for it in range(1, 31):
        b.md_advance_vv(it)
    for x, y in zip(a.state(), b.state()):
        assert np.array_equal(x, y)
    a.close()
    b.close()
