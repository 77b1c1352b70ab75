"""How the mixed form adds the forces of bonds and angles up: an atom's terms are
rounded to the accumulator's step together, not one by one."""
import numpy as np
import pytest

import ommhip

pytestmark = pytest.mark.gpu

STEP = 2.0**-32


def _stars(count, arms, seed):
    """Molecules of a centre and its arms: bonds to the centre, an angle per pair of
    arms, no nonbonded interaction."""
    n = arms + 1
    rng = np.random.default_rng(seed)
    f = ommhip.NonbondedForce()
    f.set_nonbonded_method("CutoffPeriodic")
    f.set_cutoff_distance(0.9)
    for _ in range(count * n):
        f.add_particle(0.0, 0.3, 0.0)
    centres = rng.uniform(0.0, 4.0, (count, 1, 3))
    d = rng.normal(size=(count, arms, 3))
    pos = np.concatenate([centres, centres + 0.15 * d / np.linalg.norm(d, axis=2, keepdims=True)], 1).reshape(-1, 3)
    first = n * np.arange(count)
    bonds = np.array([(c, c + a) for c in first for a in range(1, n)], np.int32)
    angles = np.array([(c + a, c, c + b) for c in first for a in range(1, n) for b in range(a + 1, n)], np.int32)
    bond_params = np.stack([rng.uniform(0.1, 0.2, len(bonds)), rng.uniform(10.0, 100.0, len(bonds))], 1)
    angle_params = np.stack([rng.uniform(1.5, 2.5, len(angles)), rng.uniform(0.1, 1.0, len(angles))], 1)
    return ommhip.WaterSystem(f, pos, 4.0 * np.eye(3), np.full(count * n, 10.0), bonds, bond_params, angles, angle_params)


@pytest.mark.parametrize("count", [1, 42, 43, 200])
def test_a_molecules_terms_are_rounded_together(count):
    # Against the plain FP64 form (forces of about 10 kJ/mol/nm, rounded at 1e-15): a
    # step per atom component, which a molecule whose terms two workgroups share
    # uses up with half a step from each.
    s = _stars(count, 3, seed=7)
    mixed = ommhip.Context(s, precision=ommhip.PRECISION_MIXED).get_state()["forces"]
    ref = ommhip.Context(s, precision=ommhip.PRECISION_DOUBLE).get_state()["forces"]
    off = np.abs(mixed - ref).max() / STEP
    print(count, off)
    assert off <= 1.001


def _pulled(length, places):
    """An atom with one bond, k = 1e9, to an atom at each of the given places about it."""
    n = len(places)
    f = ommhip.NonbondedForce()
    f.set_nonbonded_method("CutoffPeriodic")
    f.set_cutoff_distance(0.9)
    for _ in range(n + 1):
        f.add_particle(0.0, 0.3, 0.0)
    pos = np.array([[3.0, 3.0, 3.0]] + [[3.0 + x, 3.0 + y, 3.0] for x, y in places])
    bonds = np.array([(0, a) for a in range(1, n + 1)], np.int32)
    s = ommhip.WaterSystem(f, pos, 6.0 * np.eye(3), np.full(n + 1, 10.0), bonds, np.tile([length, 1e9], (n, 1)),
                           np.zeros((0, 3), np.int32), np.zeros((0, 2)))
    return ommhip.Context(s)


def test_the_range_is_that_of_an_atoms_whole_force():
    # The accumulators hold 2.1e9.  Three bonds pull with 0.9e9 each along x: 2.7e9 is reported.
    with pytest.raises(ommhip.OmmError) as e:
        _pulled(0.1, [(1.0, -0.2), (1.0, 0.0), (1.0, 0.2)]).get_state()
    assert e.value.status == ommhip.STATUS_CODES["OVERFLOW"]
    # Two of 0.9e9 against one another cancel; each partner keeps its own (1e-15 of it).
    f = _pulled(0.1, [(1.0, 0.0), (-1.0, 0.0)]).get_state()["forces"]
    assert np.abs(f - np.array([[0.0, 0, 0], [-0.9e9, 0, 0], [0.9e9, 0, 0]])).max() <= 1e-6
