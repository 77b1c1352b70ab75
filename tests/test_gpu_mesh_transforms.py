"""The mesh's matrix-core transforms (short axes, and up to 128 points with a
large prime factor) and the staged passes, at the sizes where a tile, a padded
step or the dispatch can go wrong: single tiles, remainders of 4, 8 and 16,
primes, the 64 / 65 point change of workgroup (and of path in FP64), the 120 /
121 and the 128 / 129 point changes of path."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import force_rms_rel, water

pytestmark = pytest.mark.gpu

GRIDS = [(5, 6, 7), (16, 17, 8), (31, 33, 15), (64, 9, 65), (65, 64, 11), (13, 128, 30), (127, 14, 19), (12, 21, 128), (67, 9, 14),
         (129, 10, 17), (11, 130, 16), (9, 18, 131)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("tilt", [False, True])
def test_charge_mesh_fp64(grid, tilt):
    # The charge mesh's own bars: energy and forces to 1e-12, derivatives to
    # 1e-11 relative (FP64 rounding of either transform is about 1e-15).
    rng = np.random.default_rng(sum(grid) + tilt)
    box = np.diag([2.0, 2.3, 1.9])
    if tilt:
        box[1, 0], box[2, 0], box[2, 1] = 0.6, -0.4, 0.5
    pos, q = rng.uniform(-1.0, 3.0, size=(120, 3)), rng.normal(scale=0.5, size=120)
    mesh = ommhip.PmeCache()
    f = np.zeros((120, 3))
    e = mesh.evaluate_charges(pos, q, box, (2.9, grid), f)
    f_ref, e_ref = orc.pme_mesh(pos, q, box, 2.9, grid)
    d = np.zeros(120)
    mesh.charge_derivatives(pos, q, box, (2.9, grid), np.arange(120), d)
    d_ref = orc.pme_charge_derivatives(pos, q, box, 2.9, grid)
    print(grid, abs(e - e_ref) / abs(e_ref), force_rms_rel(f, f_ref), np.abs(d - d_ref).max() / np.abs(d_ref).max())
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
    assert force_rms_rel(f, f_ref) <= 1e-12
    assert np.abs(d - d_ref).max() <= 1e-11 * np.abs(d_ref).max()


def _water(grid, seed):
    s = ommhip.water_system(300, 2.1, seed)
    s.nonbonded.set_pme_parameters(2.920290, *grid)
    return s


@pytest.mark.parametrize("grid", [(19, 19, 19), (17, 24, 33), (64, 20, 65), (20, 65, 18), (23, 19, 120), (23, 19, 121),
                                  (19, 127, 21), (129, 19, 20)])
def test_step_forces_fp32(grid):
    # The step's FP32 mesh, through the velocity of one step from rest without
    # noise or bonded terms: the mixed form's force bar, 2e-6.
    s = _water(grid, 17)
    s.bonds, s.bond_params = np.zeros((0, 2), np.int32), np.zeros((0, 2))
    s.angles, s.angle_params = np.zeros((0, 3), np.int32), np.zeros((0, 2))
    c = ommhip.Context(s, temperature=0.0, friction=0.0, step_size=0.001)
    c.set_velocities(np.zeros_like(s.positions))
    c.step(1)
    f = c.get_state()["velocities"] * s.masses[:, None] / 0.001
    f_ref = orc.nb_evaluate(s.nonbonded.desc(), s.positions, s.box)[0]
    print(grid, force_rms_rel(f, f_ref))
    assert force_rms_rel(f, f_ref) <= 2e-6


def test_batch_of_both_paths_matches_lone_contexts():
    # One replica beyond 128 points (staged passes) between two within: the
    # rule is each system's own, so a replica steps as it does alone.
    systems = [_water((19, 20, 21), 31), _water((130, 19, 18), 32), _water((66, 18, 25), 33)]
    batch = ommhip.Batch(systems, temperature=300.0, friction=1.0, seeds=[4, 5, 6])
    for r, s in enumerate(systems):
        batch.set_velocities(r, np.zeros_like(s.positions))
    batch.step(12)
    for r, s in enumerate(systems):
        lone = ommhip.Context(s, temperature=300.0, friction=1.0, seed=4 + r)
        lone.set_velocities(np.zeros_like(s.positions))
        lone.step(12)
        a, b = batch.get_state(r), lone.get_state()
        assert np.array_equal(a["positions"], b["positions"])
        assert np.array_equal(a["forces"], b["forces"])
