"""The resident form of the operator with arrays that are not one allocation of the
device: arrays that are too short are an error before any kernel uses them, page-locked
host memory is copied."""
import ctypes as C

import numpy as np
import pytest

import ommhip
from helpers import DeviceArray, hip_runtime, water

pytestmark = pytest.mark.gpu

PRECISIONS = [ommhip.PRECISION_MIXED, ommhip.PRECISION_DOUBLE]


@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("short", ["positions", "forces"])
def test_short_device_arrays_are_refused(precision, short):
    s = water(1000, 3.1, seed=85)
    op = ommhip.GpuNonbondedForce(s.nonbonded, precision)
    op.initialize(s.box)
    e_ref = op.calc_forces_and_energy(s.positions, s.box)[1]
    hip = hip_runtime()
    half = len(s.positions) // 2
    pos, forces = DeviceArray(hip, s.positions), DeviceArray(hip, np.zeros_like(s.positions))
    cut = DeviceArray(hip, s.positions[:half])
    try:
        with pytest.raises(ommhip.OmmError):
            if short == "positions":
                op.calc_forces_and_energy_device(cut.p, s.box, forces.p)
            else:
                op.calc_forces_and_energy_device(pos.p, s.box, cut.p)
        assert np.array_equal(cut.get(), s.positions[:half])  # nothing was written
        e, _ = op.calc_forces_and_energy_device(pos.p, s.box, forces.p)
        assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
    finally:
        for a in (pos, forces, cut):
            a.free()


@pytest.mark.parametrize("precision", PRECISIONS)
def test_page_locked_arrays(precision):
    s = water(1000, 3.1, seed=86)
    op = ommhip.GpuNonbondedForce(s.nonbonded, precision)
    op.initialize(s.box)
    f_ref, e_ref = op.calc_forces_and_energy(s.positions, s.box)
    hip = hip_runtime()
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    at = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(at), 2 * s.positions.nbytes, 0) == 0
    try:
        both = np.frombuffer((C.c_double * (2 * s.positions.size)).from_address(at.value)).reshape(2, -1, 3)
        both[0], both[1] = s.positions, 0.0
        e, _ = op.calc_forces_and_energy_device(at, s.box, C.c_void_p(at.value + s.positions.nbytes))
        assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
        assert np.abs(both[1] - f_ref).max() <= 1e-12 * np.abs(f_ref).max()
    finally:
        hip.hipHostFree(at)
