"""The force launches' list rows: capacities that are not whole groups of a team's lanes, lists that
fill them and lists of a word or none, in every branch-free loop, against the oracle."""
import sys

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd._abi import FM_PREC_FP64, FM_PREC_MIXED
from flowmol_amd.md import MDContext
from oracle.oracle import Oracle
from tests.helpers import rel_force_err

pytestmark = pytest.mark.gpu
TOL = {FM_PREC_FP64: 1e-12, FM_PREC_MIXED: 1e-5}


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("precision", [FM_PREC_FP64, FM_PREC_MIXED])
@pytest.mark.parametrize("brick", [(1, 1, 1), (3, 3, 3)])     # teams of lanes, and one lane a molecule
@pytest.mark.parametrize("extra", [0, 1, 4, 9])               # entries the capacity has beyond the longest list
def test_rows_at_the_capacity(precision, brick, extra):
    p, r, v = config.config_fcc((6, 6, 6), 0.8, 2.5, seed=41, tplot=2, precision=precision)
    rng = np.random.default_rng(3)
    r = r + rng.uniform(-0.1, 0.1, r.shape)
    r = r[(r[:, 0] < 1.5) | (rng.uniform(size=r.shape[0]) < 0.02)]      # a slab, and a few molecules alone
    v = v[:r.shape[0]] * 0.0
    L = np.array([p.domain[d] for d in range(3)])
    r = np.where(r < -0.5 * L, r + L, np.where(r >= 0.5 * L, r - L, r))
    d = r[:, None] - r[None]
    d -= L * np.round(d / L)
    longest = int(((d * d).sum(-1) < 2.8 ** 2).sum(1).max()) - 1
    p.max_neighbours = longest + extra
    p.brick[0], p.brick[1], p.brick[2] = brick
    say(f"case: {r.shape[0]} LJ, longest list {longest}, room for {longest + extra}, brick {brick}, precision {precision}")
    o, g = Oracle(p, r, v), MDContext(p, r, v)
    o.setup()
    g.setup(0)
    for it in (0, 1):   # a record step and a step without tallies
        o.compute_forces(it)
        g.simulation_compute_forces(it)
        assert rel_force_err(g.state()[2], o.state()[2], o.force_scale()) < TOL[precision]
    g.close()
