"""Host-side logic that needs no GPU: the brick-shape candidates of the tuner."""
import itertools

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd._abi import FM_PREC_MIXED, iptr
from flowmol_amd._lib import check, load
from flowmol_amd.md import FB_BLOCK, brick_candidates, default_brick


@pytest.mark.parametrize("ncells,nmol", [((39, 39, 39), 1048576), ((4, 4, 4), 2048), ((9, 9, 9), 2048),
                                         ((3, 3, 3), 500), ((12, 5, 7), 30000)])
def test_brick_candidates_fit_a_workgroup_pass_and_rank_by_halo(ncells, nmol):
    occ = max(1.0, nmol / float(np.prod(ncells)))
    got = brick_candidates(ncells, nmol, max_candidates=6)
    assert 1 <= len(got) <= 6
    eff = [np.prod(b) / np.prod([x + 2 for x in b]) for b in got]
    assert eff == sorted(eff, reverse=True)
    for b in got:
        assert all(1 <= b[d] <= min(ncells[d], 12) for d in range(3))
        assert np.prod(b) == 1 or np.prod(b) * occ <= FB_BLOCK * 15 / 16
    # brute force: no admissible shape has less halo per cell than the first candidate
    best = max(np.prod(b) / np.prod([x + 2 for x in b])
               for b in itertools.product(*[range(1, min(n, 12) + 1) for n in ncells])
               if np.prod(b) == 1 or np.prod(b) * occ <= FB_BLOCK * 15 / 16)
    assert abs(eff[0] - best) < 1e-15


def test_brick_candidates_at_the_1m_workload():
    # 17.7 molecules per cell: 27 cells fit one pass of 480 threads, 3x3x3 has the least halo
    assert brick_candidates((39, 39, 39), 1048576, 1) == [(3, 3, 3)]


def test_random_walk_chains():
    """Seeded random-walk chains: raw walks have every bond exactly 0.97 long (minimum image);
    after the overlap relaxation of the initial state no two non-bonded beads are closer than
    0.8 and every bond is within 0.05 of 0.97; beads inside the box; the same chains for the
    same seed."""
    from scipy.spatial import cKDTree

    from flowmol_amd import config

    p, r, v, mt, mono = config.config_polymer(nunits=(8, 8, 8), init="random_walk", seed=9)
    L = np.array([p.domain[0], p.domain[1], p.domain[2]])
    n = r.shape[0]
    assert n == 2048 and np.all(r >= -0.5 * L) and np.all(r < 0.5 * L)
    raw = config.random_walk_chains(L, n // 8, 8, 9)
    bonded = (np.arange(n - 1) % 8) != 7

    def bonds(x):
        d = x[1:] - x[:-1]
        d -= L * np.round(d / L)
        return np.linalg.norm(d, axis=1)[bonded]

    assert np.abs(bonds(raw) - 0.97).max() < 1e-12
    assert np.abs(bonds(r) - 0.97).max() <= 0.05
    pairs = cKDTree(r + 0.5 * L, boxsize=L).query_pairs(0.8, output_type="ndarray")
    close = [(i, j) for i, j in pairs if not (j == i + 1 and i % 8 != 7)]
    assert not close
    chain, sub, funcy, bflag = mono
    assert list(sub[:8]) == list(range(1, 9)) and list(funcy[:8]) == [1, 2, 2, 2, 2, 2, 2, 1]
    _, r2, _, _, _ = config.config_polymer(nunits=(8, 8, 8), init="random_walk", seed=9)
    assert np.array_equal(r, r2)


def layout(p, nmol, capacity=0, compute_units=0):
    """(brick, lanes per molecule) that a context of these parameters gets."""
    brick, team = np.zeros(3, np.int32), np.zeros(1, np.int32)
    check(load().fm_default_layout(p, nmol, capacity, compute_units, iptr(brick), iptr(team)))
    return tuple(int(x) for x in brick), int(team[0])


@pytest.mark.parametrize("density,lanes", [(0.8, 8), (1.6, 16)])   # 73 and 147 expected entries
def test_lanes_keep_the_list_offsets_within_32_bits(density, lanes):
    """A lane's place in its team's rows of the list is a 32-bit byte offset: however large the capacity
    that fm_init takes (below 2^27), lanes x capacity x 8 bytes are at most 2^32."""
    p, r, _ = config.config_fcc((8, 8, 8), 0.4, 2.5, seed=1, tplot=10)
    p.density = density
    p.brick[0] = p.brick[1] = p.brick[2] = 1
    nmol = r.shape[0]                      # 2,048 in 6^3 cells: ten a brick
    assert layout(p, nmol)[1] == lanes
    for capacity in (2 ** 24, 2 ** 25, 2 ** 25 + 1, 2 ** 26, 2 ** 26 + 1, 2 ** 27 - 1):
        team = layout(p, nmol, capacity)[1]
        assert 1 <= team <= lanes and team * capacity * 8 <= 2 ** 32
        assert team == lanes or 2 * team * capacity * 8 > 2 ** 32


def test_default_bricks_are_as_many_as_the_device_runs_at_once():
    """108,000 molecules in 18^3 cells: the largest bricks (24 cells) are too few for the 512 workgroups of
    256 CUs, which get smaller ones, and enough for a partition of 32 or 64 CUs, which keeps them."""
    p, r, _ = config.config_fcc((30, 30, 30), 0.8, 2.5, seed=1, tplot=10)
    cells, bricks = {}, {}
    for cus in (32, 64, 256):
        shape = layout(p, r.shape[0], compute_units=cus)[0]
        cells[cus], bricks[cus] = np.prod(shape), np.prod([-(-18 // b) for b in shape])
    assert cells[32] == cells[64] == 24
    assert cells[256] < 24 and 400 <= bricks[256] <= 512


@pytest.mark.parametrize("units,density,rc", [((8, 8, 8), 0.8, 2.5), ((11, 13, 9), 0.8, 2.5), ((16, 16, 16), 0.8, 2.5),
                                              ((30, 30, 30), 0.8, 2.5), ((24, 24, 24), 0.8, 4.0), ((64, 64, 64), 0.8, 2.5),
                                              ((12, 12, 12), 0.8, 1.1225)])
@pytest.mark.parametrize("mixed", [False, True])
def test_the_tuner_times_the_default_brick(units, density, rc, mixed):
    p, r, _ = config.config_fcc(units, density, rc, seed=1, tplot=10, precision=FM_PREC_MIXED if mixed else 0)
    nmol, cells = r.shape[0], [int(p.domain[d] // (rc + 0.3)) for d in range(3)]
    default = layout(p, nmol)[0]
    assert default_brick(p, nmol) == default
    for k in (1, 2, 3, 6):
        got = brick_candidates(cells, nmol, k, default)
        assert default in got and len(got) == k == len(set(got))
        if not mixed:
            assert got == brick_candidates(cells, nmol, k)


@pytest.mark.parametrize("units,density,rc", [(8, 0.8, 1.1225), (12, 0.8, 1.1225), (20, 0.8, 1.1225), (12, 0.8, 2.5),
                                              (16, 0.8, 2.5), (20, 0.8, 2.5), (30, 0.8, 2.5), (20, 0.2, 2.5), (13, 0.8, 4.0)])
def test_default_bricks_do_not_multiply_the_work_of_a_batch(units, density, rc):
    """Small bricks let a lone small domain use the whole device, but a batch in one launch costs what all
    bricks stage together: that stays near the least of any shape (300: a workgroup's own cost in staged
    molecules)."""
    p, r, _ = config.config_fcc((units,) * 3, density, rc, seed=1, tplot=10)
    nc = [int(p.domain[d] // (rc + 0.3)) for d in range(3)]
    occ = max(1.0, r.shape[0] / np.prod(nc))

    def work(b):
        return np.prod([-(-n // x) for n, x in zip(nc, b)]) * (np.prod([x + 2 for x in b]) * occ + 300.0)

    least = min(work(b) for b in itertools.product(*[range(1, min(n, 12) + 1) for n in nc])
                if np.prod(b) == 1 or np.prod(b) * occ <= FB_BLOCK * 15 / 16)
    assert work(layout(p, r.shape[0])[0]) <= max(1.4 * least, least + 80000.0) * (1 + 1e-12)
