"""Teams of lanes per molecule in the force launches: bricks of one cell up to 27, which give
teams of eight lanes down to one, on steps with and without each tally, against the oracle."""
import sys

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd.md import MDContext
from oracle.oracle import Oracle
from tests.helpers import equilibrated, rel_force_err

pytestmark = pytest.mark.gpu
TOL = 1e-12


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def liquid():
    return equilibrated(lambda: config.config_fcc((8, 8, 8), 0.8, 2.5, seed=17, tplot=10), 150)


@pytest.mark.parametrize("brick", [(1, 1, 1), (2, 1, 1), (2, 2, 1), (3, 3, 3)])   # 32, 64, 128, 864 molecules
@pytest.mark.parametrize("tally", ["none", "planes 4", "planes 16", "tensor"])     # 3 slots a molecule, ranges
def test_forces_and_tallies(liquid, brick, tally):
    base, r, v, a = liquid
    p = type(base).from_buffer_copy(base)
    p.tplot, p.teval = 4, 2
    p.brick[0], p.brick[1], p.brick[2] = brick
    if tally.startswith("planes"):
        p.vflux_outflag, p.nplanes = 2, int(tally.split()[1])
        p.planespacing = p.domain[1] / p.nplanes
    p.pressure_outflag = 1 if tally == "tensor" else 0
    say(f"case: 2048 LJ, brick {brick}, tally {tally}")
    o, g = Oracle(p, r, v, a), MDContext(p, r, v, a)
    o.setup()
    g.setup(1)
    for it in (0, 1, 2):   # a record step, a step without tallies, a virial step
        if p.vflux_outflag:
            o.reset_mop()
            g.reset_mop()
        o.compute_forces(it)
        g.simulation_compute_forces(it)
        assert rel_force_err(g.state()[2], o.state()[2], o.force_scale()) < TOL
        if it != 1:
            for ref, got in list(zip(o.molecular(), g.molecular()))[it // 2:]:   # (virial steps: no PE)
                assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()
        if it == 0 and p.vflux_outflag:
            assert np.abs(g.mop() - o.mop()).max() <= 10 * TOL * np.abs(o.mop()).max()
        if it == 0 and p.pressure_outflag:
            assert np.abs(g.rfmol() - o.rfmol()).max() <= 10 * TOL * np.abs(o.rfmol()).max()
    g.close()


@pytest.mark.parametrize("capacity", [0, 2 ** 26 + 1])   # 16 lanes, and 4 where 8 would pass 32-bit offsets
@pytest.mark.parametrize("it", [0, 1])                   # a record step, a step without tallies
def test_sixteen_lanes_and_a_capacity_beyond_32_bit_offsets(capacity, it):
    import torch

    if capacity and torch.cuda.mem_get_info()[0] < 60 * 2 ** 30:
        pytest.skip("needs 60 GiB of device memory")
    p, r, v = config.config_fcc((8, 8, 8), 0.4, 2.5, seed=19, tplot=4)
    r = r + np.random.default_rng(19).uniform(-0.2, 0.2, r.shape)
    L = np.array([p.domain[d] for d in range(3)])
    r = np.where(r < -0.5 * L, r + L, np.where(r >= 0.5 * L, r - L, r))
    p.density = 1.6                         # (the rule's expectation: 147 entries; the lists hold half)
    p.max_neighbours = 96
    p.brick[0] = p.brick[1] = p.brick[2] = 1
    say(f"case: 2048 LJ, bricks of ten, capacity {capacity}, step {it}")
    o, g = Oracle(p, r, v), MDContext(p, r, v, capacity=capacity)
    o.setup()
    g.setup(1)
    o.compute_forces(it)
    g.simulation_compute_forces(it)
    assert rel_force_err(g.state()[2], o.state()[2], o.force_scale()) < TOL
    if it == 0:
        for ref, got in zip(o.molecular(), g.molecular()):
            assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()
    g.close()
