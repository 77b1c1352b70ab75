"""The neighbour list's order by a workgroup per system (systems of one unit size),
with or without the bounds, against each other and the oracle."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import water

pytestmark = pytest.mark.gpu


# Below, at and above the 1,024 units of the one-workgroup list, one unit, a
# tilted box with few cells.
@pytest.mark.parametrize("molecules,edge,tilt", [(1, 1.85, 0.0), (22, 1.85, 0.3), (1024, 3.2, 0.1),
                                                 (1025, 3.2, 0.0), (2048, 3.95, 0.2),
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
    # A replica of a batch is placed by a launch of its own.
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


@pytest.mark.parametrize("molecules", [8192, 8193])
def test_units_at_the_workgroup_limit(molecules):
    # At most 8,192 units: a workgroup orders them; more: the launches of large
    # systems.
    s = water(molecules, 6.4, seed=3, cutoff=0.9)
    op = ommhip.GpuNonbondedForce(s.nonbonded)
    op.initialize(s.box)
    rng = np.random.default_rng(2)
    for _ in range(2):
        pos = s.positions + rng.normal(scale=0.01, size=s.positions.shape)
        assert op.pair_stats(pos, s.box) == orc.nb_pairs(s.nonbonded.desc(), pos, s.box)


def test_batch_whose_systems_build_on_different_steps():
    # Replicas of very different sizes and speeds: most steps rebuild some lists
    # and keep others.
    sizes = [(40, 1.9), (700, 2.9), (3, 1.85), (2100, 4.1)]
    systems = [water(m, e, seed=m, cutoff=0.9) for m, e in sizes]
    rng = np.random.default_rng(8)
    v = [rng.normal(scale=0.3 * (k + 1), size=s.positions.shape) for k, s in enumerate(systems)]
    batch = ommhip.Batch(systems, temperature=300.0, friction=1.0, seeds=[1, 2, 3, 4])
    for k in range(4):
        batch.set_velocities(k, v[k])
    batch.step(40)
    for k, s in enumerate(systems):
        lone = ommhip.Context(s, temperature=300.0, friction=1.0, seed=k + 1)
        lone.set_velocities(v[k])
        lone.step(40)
        a, b = lone.get_state(), batch.get_state(k)
        assert np.array_equal(a["positions"], b["positions"])
        assert np.array_equal(a["velocities"], b["velocities"])
