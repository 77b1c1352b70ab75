"""The list of the evaluation calls follows the box, whichever group sees a new
box first: a call that reads no list must not use up the change."""
import numpy as np
import pytest

import ommhip
from helpers import water

pytestmark = pytest.mark.gpu

DIRECT, RECIPROCAL = 1 << 0, 1 << 1


def _operator(s, precision):
    s.nonbonded.set_force_group(0)
    s.nonbonded.set_reciprocal_space_force_group(1)
    op = ommhip.GpuNonbondedForce(s.nonbonded, precision)
    op.initialize(s.box)
    return op


@pytest.mark.parametrize("precision", [ommhip.PRECISION_MIXED, ommhip.PRECISION_DOUBLE])
@pytest.mark.parametrize("first", ["both groups", "reciprocal group"])
def test_direct_call_after_the_reciprocal_group_took_a_new_box(precision, first):
    # A gap at the boundary, wider than the list's skin, closes with the
    # positions as they are: pairs across it come into range that the old list lacks.
    s = water(1000, 3.1, seed=91)
    box, s.box = s.box, s.box + 0.2 * np.eye(3)
    op = _operator(s, precision)
    if first == "both groups":
        op.calc_forces_and_energy_groups(s.positions, s.box, DIRECT | RECIPROCAL)
    else:  # the first list is built after a reciprocal call in the old box
        op.calc_forces_and_energy_groups(s.positions, s.box, RECIPROCAL)
    op.calc_forces_and_energy_groups(s.positions, box, RECIPROCAL)
    f, e = op.calc_forces_and_energy_groups(s.positions, box, DIRECT)
    f_ref, e_ref = _operator(s, precision).calc_forces_and_energy_groups(s.positions, box, DIRECT)
    assert op.pair_stats(s.positions, box) == _operator(s, precision).pair_stats(s.positions, box)
    # Lists in one order: the mixed form's sums agree in every bit, FP64 atomics to rounding.
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
    assert np.abs(f - f_ref).max() <= 1e-12 * np.abs(f_ref).max()
