"""How the mixed form adds the pair forces up: steps of 2^-32 kJ/mol/nm on either
side of a pair, and a range that is the whole force's."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import lj_pair_system

pytestmark = pytest.mark.gpu

STEP = 2.0**-32


@pytest.mark.parametrize("eps", [1e-6, 1e-5, 1e-4, 1e-3])
def test_weak_forces_keep_the_accumulators_step(eps):
    # One pair: each atom's force is one sum, off by a step at most (rounded on
    # one side, cut on the other) beside the FP32 arithmetic.  That is below 3e-6:
    # coordinates off by 2^-25 of 0.5 nm at r > 0.4 nm through a power of 14, and
    # about ten roundings.
    f, pos, box = lj_pair_system(np.diag([3.0, 4.0, 5.0]))
    for a in range(2):
        q, sigma, _ = f.particles[a]
        f.particles[a] = (q, sigma, eps)
    rng = np.random.default_rng(5)
    op = ommhip.GpuNonbondedForce(f)
    op.initialize(box)
    worst = 0.0
    for _ in range(40):
        d = rng.normal(size=3)
        pos[1] = pos[0] + rng.uniform(0.4, 0.9) * d / np.linalg.norm(d)
        ref = orc.nb_evaluate(f.desc(), pos, box)[0]
        worst = max(worst, ((np.abs(op.calc_forces(pos, box) - ref) - 3e-6 * np.abs(ref).max()) / STEP).max())
    print(eps, worst)
    assert worst <= 1.0


def test_pair_energies_are_rounded_not_cut():
    # Charges of one sign: every tile's energy is positive.  Some 8,000 tiles, rounded to a
    # step each: 0.29 x sqrt(8,000) = 26 steps of scatter, of which 200 allow for several
    # deviations and for the FP64 sums (1e-15 of 1e6 kJ/mol).  Cut to a step each they
    # lose 4,000.
    rng = np.random.default_rng(8)
    f = ommhip.NonbondedForce()
    f.set_nonbonded_method("CutoffPeriodic")
    f.set_cutoff_distance(0.9)
    for _ in range(9000):
        f.add_particle(0.1, 0.3, 0.0)
    pos, box, direct = rng.uniform(0.0, 4.48, (9000, 3)), 4.48 * np.eye(3), []
    for precision in (ommhip.PRECISION_MIXED, ommhip.PRECISION_DOUBLE):
        op = ommhip.GpuNonbondedForce(f, precision)
        op.initialize(box)
        direct.append(op.energy_parts(pos, box)[0])
    print(direct, (direct[0] - direct[1]) / STEP)
    assert abs(direct[0] - direct[1]) <= 200 * STEP


def _one_against(offsets, eps):
    """An atom and partners that do not act on each other, at its position plus the offsets."""
    n = len(offsets)
    f = ommhip.NonbondedForce()
    f.set_nonbonded_method("CutoffPeriodic")
    f.set_cutoff_distance(1.0)
    f.set_use_dispersion_correction(False)
    for _ in range(n + 1):
        f.add_particle(0.0, 0.3, eps)
    for i in range(1, n + 1):
        for j in range(i + 1, n + 1):
            f.add_exception(i, j, 0.0, 0.3, 0.0)
    pos = np.vstack([[0.2, 0.2, 0.2], np.array([0.2, 0.2, 0.2]) + offsets])
    box = 3.0 * np.eye(3)
    op = ommhip.GpuNonbondedForce(f)
    op.initialize(box)
    return op, pos, box


# The LJ force at 0.1 nm with sigma 0.3 nm, per unit of epsilon.
PUSH = 24.0 / 0.1 * (2.0 * 3.0**12 - 3.0**6)


def test_force_beyond_the_range_is_reported():
    # Sixteen partners of 2.0e8 kJ/mol/nm each in one direction: no lane's sum of
    # eight leaves the accumulator's 2^31, the atom's does.
    op, pos, box = _one_against(np.tile([0.1, 0.0, 0.0], (16, 1)), 0.8)
    with pytest.raises(ommhip.OmmError) as e:
        op.calc_forces(pos, box)
    assert e.value.status == ommhip.STATUS_CODES["OVERFLOW"]


def test_large_forces_that_cancel_are_accepted():
    # Eight partners of 4.1e8 on either side: a lane's sum may leave 2^31, the
    # atom's force is small.  Coordinates off by 2^-25 of 0.5 nm at 0.1 nm: 4e-6.
    op, pos, box = _one_against(np.repeat([[0.1, 0.0, 0.0], [-0.1, 0.0, 0.0]], 8, axis=0), 1.6)
    f = op.calc_forces(pos, box)
    push = 1.6 * PUSH
    expected = np.zeros((17, 3))
    expected[1:9, 0], expected[9:, 0] = push, -push
    assert np.abs(f[1:] - expected[1:]).max() <= 1e-5 * push
    assert np.abs(f[0]).max() <= 16 * 1e-5 * push
