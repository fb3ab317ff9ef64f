"""The MOP record step's plane slots: spacings either side of half the cutoff (two slots above a
molecule, or the loop over the planes between), molecules exactly on planes and at the box's faces,
in a box whose every brick has images, against the oracle."""
import sys

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd._abi import FM_PREC_FP64, FM_PREC_MIXED
from flowmol_amd.md import MDContext
from oracle.oracle import Oracle
from tests.helpers import rel_force_err

pytestmark = pytest.mark.gpu
TOL = 1e-12


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("precision", [FM_PREC_FP64, FM_PREC_MIXED])
@pytest.mark.parametrize("brick", [(1, 1, 1), (3, 3, 3)])
@pytest.mark.parametrize("spacing", [1.2501, 1.2499, 1.9, 2.5, 4.0])
def test_plane_slots(spacing, brick, precision):
    p, r, v = config.config_fcc((6, 6, 6), 0.8, 2.5, seed=29, tplot=1, precision=precision)
    L = p.domain[1]
    p.vflux_outflag, p.planespacing, p.nplanes = 2, spacing, int(L / spacing)
    p.brick[0], p.brick[1], p.brick[2] = brick
    rng = np.random.default_rng(7)
    r = r + rng.uniform(-0.1, 0.1, r.shape)
    r = np.where(r < -0.5 * L, r + L, np.where(r >= 0.5 * L, r - L, r))
    planes = Oracle(p, r, v).planes()
    for n in range(0, r.shape[0], 5):   # one molecule in five on the plane nearest to it, or a rounding off
        k = np.abs(planes - r[n, 1]).argmin()
        if abs(planes[k] - r[n, 1]) < 0.15:
            r[n, 1] = planes[k] + rng.choice([-1e-15, 0.0, 1e-15])
    say(f"case: {r.shape[0]} LJ, {p.nplanes} planes {spacing} apart, brick {brick}, precision {precision}")
    o, g = Oracle(p, r, v), MDContext(p, r, v)
    o.setup()
    g.setup(0)
    o.reset_mop()
    g.reset_mop()
    o.compute_forces(0)
    g.simulation_compute_forces(0)
    assert rel_force_err(g.state()[2], o.state()[2], o.force_scale()) < TOL
    assert np.abs(g.mop() - o.mop()).max() <= 10 * TOL * np.abs(o.mop()).max()
    g.close()
