"""Spreads of atoms that no list has ordered: charge meshes at the limits of the
plane-wise spread, and reciprocal-only calls, on both sides of the change to
tiles (12,000 atoms)."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import water

pytestmark = pytest.mark.gpu

DIRECT, RECIPROCAL = 1 << 0, 1 << 1


# Planes of 6,144 points and more; planes times charges of 4e7 and more; each with
# few enough atoms to add directly, and with more.
@pytest.mark.parametrize("n,grid", [(12000, (8, 96, 64)), (12000, (8, 96, 65)), (12001, (8, 96, 65)), (40000, (1000, 8, 9)),
                                    (40001, (1000, 8, 9)), (70000, (24, 20, 25))])
def test_charge_mesh_at_the_limits_of_the_planes(n, grid):
    rng = np.random.default_rng(n + grid[2])
    box = np.diag([g / 10.0 for g in grid])
    box[1, 0], box[2, 1] = 0.1, -0.1
    pos = rng.uniform(-1.0, 2.0, size=(n, 3)) @ box
    q = rng.normal(scale=0.5, size=n)
    q[3::7] = 0.0
    mesh, alpha, f, d = ommhip.PmeCache(), 2.9, np.zeros((n, 3)), np.zeros(500)
    idx = rng.integers(0, n, size=500).astype(np.int32)
    e = mesh.evaluate_charges(pos, q, box, (alpha, grid), f)
    mesh.charge_derivatives(pos, q, box, (alpha, grid), idx, d)
    f_ref, e_ref = orc.pme_mesh(pos, q, box, alpha, grid)
    d_ref = orc.pme_charge_derivatives(pos, q, box, alpha, grid)[idx]
    # The charge mesh's bars: FP64 sums of every charge's contribution.
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
    assert np.sqrt(((f - f_ref) ** 2).sum() / (f_ref**2).sum()) <= 1e-12
    assert np.abs(d - d_ref).max() <= 1e-13 * 138.9 * np.abs(q).sum() * alpha


@pytest.mark.parametrize("method", ["PME", "LJPME"])
@pytest.mark.parametrize("precision", [ommhip.PRECISION_MIXED, ommhip.PRECISION_DOUBLE])
@pytest.mark.parametrize("molecules", [4000, 4001])
def test_reciprocal_calls_without_an_order(molecules, precision, method):
    # The atoms in a random order, before any list and after a list of another
    # conformation: what a full evaluation adds to the direct group's.
    s = water(molecules, 4.95, seed=5, method=method)
    s.nonbonded.set_force_group(0)
    s.nonbonded.set_reciprocal_space_force_group(1)
    op = ommhip.GpuNonbondedForce(s.nonbonded, precision)
    op.initialize(s.box)
    order = np.random.default_rng(6).permutation(molecules)
    other = np.ascontiguousarray(s.positions.reshape(-1, 3, 3)[order].reshape(-1, 3))
    first = op.calc_forces_and_energy_groups(other, s.box, RECIPROCAL)
    op.calc_forces_and_energy_groups(s.positions, s.box, DIRECT | RECIPROCAL)
    second = op.calc_forces_and_energy_groups(other, s.box, RECIPROCAL)
    both = op.calc_forces_and_energy_groups(other, s.box, DIRECT | RECIPROCAL)
    direct = op.calc_forces_and_energy_groups(other, s.box, DIRECT)
    if precision == ommhip.PRECISION_MIXED:
        # One fixed-point grid in every bit, whichever spread wrote it.
        assert np.array_equal(first[0], second[0]) and first[1] == second[1]
    scale = np.abs(both[0]).max()
    for f, e in (first, second):
        # Forces of 1e3 in steps of 2^-32, or FP64 sums.
        assert np.abs(both[0] - direct[0] - f).max() <= 1e-11 * scale
        assert abs(both[1] - direct[1] - e) <= 1e-11 * abs(e)
