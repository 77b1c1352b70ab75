"""The step's FP32 mesh against the FP64 oracle on long axes: the dense transforms
are no less accurate than transforms in stages."""
import numpy as np
import pytest

import ommhip
import oracle as orc

pytestmark = pytest.mark.gpu

# Relative RMS force error of the staged FP32 passes on the inputs below, the
# mean over the three axes (this library with the staged passes: 1.66e-6, 1.58e-6
# and 1.70e-6).  One rounding chain over 120 points has 2.5e-6.
STAGED = 1.65e-6


def _error(grid, seed):
    n, alpha = 2000, 2.92
    rng = np.random.default_rng(seed)
    box = np.diag([g / 9.0 for g in grid])
    pos, q = rng.uniform(0, 1, (n, 3)) @ box, np.where(np.arange(n) % 2 == 0, 0.7, -0.7)
    f = ommhip.NonbondedForce()
    f.set_nonbonded_method("PME")
    f.set_cutoff_distance(0.5)
    f.set_pme_parameters(alpha, *grid)
    f.set_include_direct_space(False)
    for x in q:
        f.add_particle(x, 1.0, 0.0)
    masses = np.full(n, 10.0)
    s = ommhip.WaterSystem(f, pos, box, masses, np.zeros((0, 2), np.int32), np.zeros((0, 2)),
                           np.zeros((0, 3), np.int32), np.zeros((0, 2)))
    # The mesh forces through the velocities of one step from rest without noise.
    c = ommhip.Context(s, temperature=0.0, friction=0.0, step_size=0.001)
    c.set_velocities(np.zeros_like(pos))
    c.step(1)
    forces = c.get_state()["velocities"] * masses[:, None] / 0.001
    ref = orc.pme_mesh(pos, q, box, alpha, grid)[0]
    return float(np.sqrt(((forces - ref) ** 2).sum() / (ref**2).sum()))


def test_dense_fp32_transforms_of_a_long_axis():
    errors = [np.mean([_error(np.roll((120, 12, 12), axis), seed) for seed in range(8)]) for axis in range(3)]
    print(errors)
    assert np.mean(errors) <= STAGED
