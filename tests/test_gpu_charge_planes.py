"""Charge meshes of particles in no order: the spread plane by plane, the
allocation-free mesh on the half spectrum, against the oracle's reciprocal sum."""
import numpy as np
import pytest

import ommhip
import oracle as orc
from helpers import hip_runtime as _hip
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


# Even, odd and the smallest and largest axes, tilted boxes (the points -n/2 of
# even axes are their own negatives), one particle, more than a batch of the
# plane's list, and more than the plane-wise spread takes.
@pytest.mark.parametrize("n,grid,tilt", [(1, (5, 6, 7), 0.4), (300, (20, 18, 16), 0.45), (300, (21, 15, 5), 0.3),
                                         (5000, (64, 64, 64), 0.2), (16384, (24, 20, 25), 0.0),
                                         (65536, (24, 20, 25), 0.1),
                                         (65537, (24, 20, 25), 0.35)])
def test_potentials_of_both_meshes(n, grid, tilt):
    hip = _hip()
    rng = np.random.default_rng(n + grid[0])
    box = np.array([[2.3, 0, 0], [tilt, 2.5, 0], [tilt * 0.5, -tilt, 2.7]])
    pos = rng.uniform(-3.0, 6.0, size=(n, 3))
    q = rng.normal(scale=0.5, size=n)
    q[3::7] = 0.0
    idx = rng.integers(0, n, size=max(1, min(n, 901))).astype(np.int32)
    alpha = 3.1
    out = np.zeros(len(idx))
    ommhip.PmeCache().charge_derivatives(pos, q, box, (alpha, grid), idx, out)
    got = _noalloc(hip, pos, q, box, alpha, grid, idx, np.zeros(len(idx)))
    ref = orc.pme_charge_derivatives(pos, q, box, alpha, grid)[idx]
    # FP64 sums of every charge's contribution.
    scale = 138.9 * np.abs(q).sum() * alpha
    assert np.abs(got - ref).max() <= 1e-13 * scale
    assert np.abs(out - ref).max() <= 1e-13 * scale
