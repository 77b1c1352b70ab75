"""Pair-kernel tasks of one, two or four tiles, chosen by the number of blocks of
a batch (64 and 384 are the last of one and of two): parity at both sides of
each change, and a replica's bits alone (small tasks) and beside a large one."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import energy_rel, force_rms_rel, water

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("molecules", [682, 683, 4096, 4097])
def test_forces_and_energy_at_task_sizes(molecules):
    s = water(molecules, (molecules / 33.4) ** (1.0 / 3.0), seed=molecules)
    op = ommhip.GpuNonbondedForce(s.nonbonded)
    op.initialize(s.box)
    F, E = op.calc_forces_and_energy(s.positions, s.box)
    F_ref, E_ref, parts = orc.nb_evaluate(s.nonbonded.desc(), s.positions, s.box)
    print(molecules, force_rms_rel(F, F_ref), energy_rel(E, E_ref))
    assert force_rms_rel(F, F_ref) <= 2e-6
    assert energy_rel(E, E_ref) <= 1e-6
    # The FP64 pair energies: 1e-9 of the direct-space sum of magnitudes.
    got = op.energy_parts(s.positions, s.box)
    assert abs(got[0] - parts[0]) <= 1e-9 * max(abs(parts[0]), abs(E_ref))
    assert op.pair_stats(s.positions, s.box) == orc.nb_pairs(s.nonbonded.desc(), s.positions, s.box)


def test_replica_does_not_see_the_task_size():
    small, large = water(300, 2.1, seed=5), water(4200, 5.0, seed=6)
    batch = ommhip.Batch([small, large], temperature=300.0, friction=1.0, seeds=[3, 4])
    lone = ommhip.Context(small, temperature=300.0, friction=1.0, seed=3)
    for c, args in ((batch, (0,)), (lone, ())):
        c.set_velocities(*args, np.zeros_like(small.positions))
        c.step(12)
    a, b = batch.get_state(0), lone.get_state()
    assert np.array_equal(a["positions"], b["positions"])
    assert np.array_equal(a["forces"], b["forces"])
