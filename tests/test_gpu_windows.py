"""The list build's x windows from the rows' bin tables (sixteen bins a cell): empty cells, rows and
bricks, x at the bins' edges, partial bricks, and regions large enough that the tables take fewer
bins, in both precisions, against the oracle's neighbour set."""
import sys

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd._abi import FM_PREC_FP64, FM_PREC_MIXED
from flowmol_amd.md import MDContext
from oracle.oracle import Oracle
from tests.helpers import canonical_pairs

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def filled(fill, n, seed):
    """n molecules in a box of 5^3 cells of side 2.8 (half a box for "half", rows of cells two apart
    in y and z for "rows"; for "edges" x on the edges of sixteenths of a cell and beside them,
    the cells' own faces left out: the oracle refuses an image rounded past its halo cells)."""
    rng = np.random.default_rng(seed)
    r = rng.uniform(0.0, 14.0, (n, 3))
    if fill == "half":
        r[:, 0] *= 0.5
    if fill == "rows":
        r[:, 1:] = 5.6 * rng.integers(0, 3, (n, 2)) + rng.uniform(0.0, 2.8, (n, 2))
    if fill == "edges":
        r[:, 0] = 0.175 * (16 * rng.integers(0, 5, n) + rng.integers(1, 16, n)) + rng.choice([-1e-12, -1e-15, 0.0, 1e-15, 1e-12], n)
    r -= 7.0
    return np.where(r < -7.0, r + 14.0, np.minimum(r, np.nextafter(7.0, 0.0)))


@pytest.mark.parametrize("precision", [FM_PREC_FP64, FM_PREC_MIXED])
@pytest.mark.parametrize("fill,n,brick", [
    ("all", 40, (3, 3, 3)), ("all", 1, (5, 5, 5)), ("half", 900, (2, 3, 4)), ("half", 300, (1, 5, 1)),
    ("rows", 1000, (3, 2, 1)), ("rows", 700, (5, 5, 5)), ("edges", 2400, (3, 3, 3)), ("edges", 600, (1, 2, 5)),
    ("all", 2500, (3, 3, 3)), ("all", 3000, (3, 3, 3)), ("edges", 3500, (3, 3, 3)), ("all", 5000, (3, 3, 3)),
])
def test_windows_keep_the_neighbour_set(precision, fill, n, brick):
    r = filled(fill, n, seed=n)
    p = config.make_params((14.0, 14.0, 14.0), n / 14.0 ** 3, 2.5, tplot=10)
    p.precision = precision
    p.brick[0], p.brick[1], p.brick[2] = brick
    say(f"case: {n} molecules, fill {fill}, brick {brick}, precision {precision}")
    o, g = Oracle(p, r, np.zeros_like(r)), MDContext(p, r, np.zeros_like(r))
    for x in (o, g):
        x.assign_to_cell()
    o.updateborders(1)
    o.assign_to_neighbourlist()
    g.messenger_updateborders(1)
    g.assign_to_neighbourlist()
    assert np.array_equal(canonical_pairs(*o.neighbourlist()), canonical_pairs(*g.neighbourlist()))
    g.close()


def at_faces(columns, seed):
    """Columns along x of five molecules, one beside a face of each cell, up to 2e-4 to either side: half
    a step of the list build's quantised grid and less.  Next ones are 2.8, the list radius and the side
    of a cell, apart within 4e-4."""
    rng = np.random.default_rng(seed)
    yz = np.repeat(rng.uniform(0.01, 13.99, (columns, 2)), 5, axis=0) + rng.uniform(-2e-3, 2e-3, (5 * columns, 2))
    x = 2.8 * np.tile(np.arange(5), columns) + rng.uniform(1e-6, 2e-4, 5 * columns) * rng.choice([-1.0, 1.0], 5 * columns)
    r = np.column_stack([np.where(x < 0.0, x + 14.0, x), yz]) - 7.0
    return r[rng.permutation(r.shape[0])]


@pytest.mark.parametrize("precision", [FM_PREC_FP64, FM_PREC_MIXED])
@pytest.mark.parametrize("columns,brick", [(400, (3, 3, 3)), (600, (2, 3, 4)), (300, (5, 2, 3)), (40, (1, 1, 1))])
def test_pairs_beside_the_cells_faces(precision, columns, brick):
    r = at_faces(columns, seed=columns)
    p = config.make_params((14.0, 14.0, 14.0), r.shape[0] / 14.0 ** 3, 2.5, tplot=10)
    p.precision = precision
    p.brick[0], p.brick[1], p.brick[2] = brick
    say(f"case: {r.shape[0]} molecules beside the faces, brick {brick}, precision {precision}")
    o, g = Oracle(p, r, np.zeros_like(r)), MDContext(p, r, np.zeros_like(r))
    for x in (o, g):
        x.assign_to_cell()
    o.updateborders(1)
    o.assign_to_neighbourlist()
    g.messenger_updateborders(1)
    g.assign_to_neighbourlist()
    assert np.array_equal(canonical_pairs(*o.neighbourlist()), canonical_pairs(*g.neighbourlist()))
    g.close()


# Cells shorter than the list radius: the reference looks at the 27 cells around a molecule's own, so
# a pair nearer than the radius whose cells are two apart is in no list.
@pytest.mark.parametrize("precision", [FM_PREC_FP64, FM_PREC_MIXED])
@pytest.mark.parametrize("n,brick", [(700, (1, 1, 1)), (900, (2, 1, 1)), (1600, (5, 1, 2)), (1500, (3, 1, 1)),
                                     (2500, (3, 3, 3)), (3000, (5, 2, 2))])
def test_unequal_skins(precision, n, brick):
    rng = np.random.default_rng(n)
    L = np.array([12.5, 14.75, 14.75])      # 5 cells of 2.5, 2.95 and 2.95; list radius 2.8
    r = rng.uniform(-0.5, 0.5, (n, 3)) * L
    p = config.make_params(L, n / L.prod(), 2.5, tplot=10)
    p.precision = precision
    for d, skin in enumerate((0.0, 0.45, 0.45)):
        p.delta_rneighbr[d] = skin
    p.brick[0], p.brick[1], p.brick[2] = brick
    say(f"case: {n} molecules, cells of 2.5, radius 2.8, brick {brick}, precision {precision}")
    o, g = Oracle(p, r, np.zeros_like(r)), MDContext(p, r, np.zeros_like(r))
    for x in (o, g):
        x.assign_to_cell()
    o.updateborders(1)
    o.assign_to_neighbourlist()
    g.messenger_updateborders(1)
    g.assign_to_neighbourlist()
    assert np.array_equal(canonical_pairs(*o.neighbourlist()), canonical_pairs(*g.neighbourlist()))
    g.close()


@pytest.mark.parametrize("brick", [(1, 1, 1), (3, 2, 2), (7, 1, 3), (7, 9, 4)])
def test_bond_length_beyond_the_cells(brick):
    p, r, v, moltype, mono = config.config_polymer((6, 8, 6), seed=12)
    p.rcutoff = config.WCA_CUT              # cells of 1.436 and 1.49, list radius R_0 = 1.5
    rng = np.random.default_rng(7)
    r = r + rng.uniform(-1.0, 1.0, r.shape) * (0.15, 0.03, 0.03)
    L = np.array([p.domain[d] for d in range(3)])
    r = np.where(r < -0.5 * L, r + L, np.where(r >= 0.5 * L, r - L, r))
    p.brick[0], p.brick[1], p.brick[2] = brick
    say(f"case: chains, cells of 1.44, radius 1.5, brick {brick}")
    o, g = Oracle(p, r, v), MDContext(p, r, v)
    for x in (o, g):
        x.set_moltype(moltype)
        x.set_monomers(*mono)
        x.assign_to_cell()
    o.updateborders(1)
    o.assign_to_neighbourlist()
    g.messenger_updateborders(1)
    g.assign_to_neighbourlist()
    assert np.array_equal(canonical_pairs(*o.neighbourlist()), canonical_pairs(*g.neighbourlist()))
    canon = lambda b, s: sorted((i, int(x), int(y)) for i in range(b.shape[0]) for x, y in zip(b[i], s[i]) if x >= 0)
    assert canon(*o.bonds()) == canon(*g.bonds())
    g.close()


# The list build by matrix tiles (FP64, small bricks): runs whose windows are empty, end within an octet, and
# take more than four blocks of 32 candidates, lists longer than the capacity first allocated.
@pytest.mark.parametrize("side", [2.8, 2.9])     # of a cell: the list radius itself, and more
@pytest.mark.parametrize("n,rows,brick", [(15, 1, (1, 1, 1)), (17, 1, (3, 1, 1)), (130, 1, (1, 1, 1)), (600, 1, (1, 1, 1)),
                                          (1200, 1, (1, 1, 1)), (1000, 2, (2, 1, 1)), (1600, 3, (1, 2, 1))])
def test_tiles_with_long_and_short_runs(n, rows, brick, side):
    rng = np.random.default_rng(n)
    L = 5.0 * side
    r = rng.uniform(0.0, L, (n, 3))
    r[:, 1:] = side * (rng.integers(0, rows, (n, 2)) + rng.uniform(0.01, 0.99, (n, 2)))
    r -= 0.5 * L
    p = config.make_params((L, L, L), n / L ** 3, 2.5, tplot=10)
    p.brick[0], p.brick[1], p.brick[2] = brick
    say(f"case: {n} molecules in {rows}^2 rows of cells of {side}, brick {brick}")
    o, g = Oracle(p, r, np.zeros_like(r)), MDContext(p, r, np.zeros_like(r))
    for x in (o, g):
        x.assign_to_cell()
    o.updateborders(1)
    o.assign_to_neighbourlist()
    g.messenger_updateborders(1)
    g.assign_to_neighbourlist()
    assert np.array_equal(canonical_pairs(*o.neighbourlist()), canonical_pairs(*g.neighbourlist()))
    g.close()
