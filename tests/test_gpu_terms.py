"""Exceptions, bonds and angles behind the pair kernel, at the edges of their
tiles (256 atoms, four waves of 64 terms of one kind), against the oracle."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import water

pytestmark = pytest.mark.gpu


# Bonds fill a wave at 32 molecules; without bonds and angles the atoms fill a
# tile at 85.
@pytest.mark.parametrize("molecules,bonded", [(1, True), (32, True), (33, True), (97, True), (85, False), (86, False)])
def test_water_terms_at_tile_edges(molecules, bonded):
    s = water(molecules, 2.2, seed=molecules)
    if not bonded:
        s.bonds, s.bond_params = np.zeros((0, 2), np.int32), np.zeros((0, 2))
        s.angles, s.angle_params = np.zeros((0, 3), np.int32), np.zeros((0, 2))
    # FP64 against FP64: sums of some hundred terms and mesh transforms.
    state = ommhip.Context(s, temperature=0.0, friction=0.0, precision=ommhip.PRECISION_DOUBLE).get_state()
    f, e = orc.water_energy_forces(s)
    assert np.abs(state["forces"] - f).max() <= 1e-10 * np.abs(f).max()
    assert abs(state["potential_energy"] - e) <= 1e-10 * abs(e) + 1e-8


def _chain(n, seed):
    # A chain folded at random, with bonds between far particles too: terms of one
    # particle lie in several tiles.  No nonbonded interaction.
    rng = np.random.default_rng(seed)
    f = ommhip.NonbondedForce(method=ommhip.NO_CUTOFF)
    for _ in range(n):
        f.add_particle(0.0, 0.3, 0.0)
    pos = np.cumsum(rng.normal(size=(n, 3)) * 0.1, axis=0)
    near = np.array([(i, i + 1) for i in range(n - 1)], np.int32)
    far = rng.integers(0, n, size=(n, 2)).astype(np.int32)
    far = far[far[:, 0] != far[:, 1]]
    bonds = np.concatenate([near, far])
    angles = np.array([(i, i + 1, i + 2) for i in range(n - 2)], np.int32)
    return ommhip.WaterSystem(f, pos, np.eye(3) * 50.0, np.full(n, 12.0), bonds,
                              np.stack([rng.uniform(0.1, 0.2, len(bonds)), rng.uniform(1e3, 2e3, len(bonds))], 1),
                              angles, np.stack([rng.uniform(1.5, 2.5, len(angles)),
                                                rng.uniform(50.0, 100.0, len(angles))], 1))


@pytest.mark.parametrize("precision", [ommhip.PRECISION_MIXED, ommhip.PRECISION_DOUBLE])
def test_terms_of_a_long_chain(precision):
    s = _chain(700, 3)
    c = ommhip.Context(s, temperature=0.0, friction=0.0, precision=precision)
    state = c.get_state()
    fb, eb = orc.harmonic_bonds(s.bonds, s.bond_params, s.positions)
    fa, ea = orc.harmonic_angles(s.angles, s.angle_params, s.positions)
    f, e = fb + fa, eb + ea
    # Mixed: every term's component is cut to 2^-32 (fewer than 40 a particle);
    # both: FP64 rounding, an angle's by its sine (above 1e-2 here).
    assert np.abs(state["forces"] - f).max() <= 1e-11 * np.abs(f).max() + 1e-8
    assert abs(state["potential_energy"] - e) <= 1e-11 * abs(e)
