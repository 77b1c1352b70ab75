"""The neighbour list's order by one workgroup (small systems of one unit size)
and by the launches of larger systems, against each other and the oracle."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import water

pytestmark = pytest.mark.gpu


# Below, at and above 2,048 units (whose last wave of blocks is partial), one
# unit, and a tilted box with few cells.
@pytest.mark.parametrize("molecules,edge,tilt", [(1, 1.85, 0.0), (22, 1.85, 0.3), (1025, 3.2, 0.0), (2048, 3.95, 0.2),
                                                 (2049, 3.95, 0.2)])
def test_pairs_and_steps_at_the_size_limits(molecules, edge, tilt):
    s = water(molecules, edge, seed=molecules, cutoff=0.9)
    s.box[2, 0] = tilt * edge
    op = ommhip.GpuNonbondedForce(s.nonbonded)
    op.initialize(s.box)
    desc = s.nonbonded.desc()
    rng = np.random.default_rng(2)
    for _ in range(3):
        pos = s.positions + rng.normal(scale=0.01, size=s.positions.shape)
        assert op.pair_stats(pos, s.box) == orc.nb_pairs(desc, pos, s.box)
    # A replica of a batch is ordered by the launches of larger systems.
    lone = ommhip.Context(s, temperature=300.0, friction=1.0, seed=5)
    batch = ommhip.Batch([s, s], temperature=300.0, friction=1.0, seeds=[5, 6])
    v = rng.normal(scale=0.5, size=s.positions.shape)
    lone.set_velocities(v)
    batch.set_velocities(0, v)
    lone.step(25)
    batch.step(25)
    a, b = lone.get_state(), batch.get_state(0)
    assert np.array_equal(a["positions"], b["positions"])
    assert np.array_equal(a["velocities"], b["velocities"])
