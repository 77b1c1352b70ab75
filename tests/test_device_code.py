"""Properties of the device code that no run shows reliably, read from its sources."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openmm-rs_amd", "csrc")
SOURCES = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))


def test_waves_hand_values_over_behind_a_fence():
    # A wave barrier alone orders no memory: it stands in one place, behind its fence.
    found = []
    for path in SOURCES:
        lines = open(path).read().splitlines()
        found += [(os.path.basename(path), lines[k - 1]) for k, line in enumerate(lines) if "amdgcn_wave_barrier" in line]
    assert [name for name, _ in found] == ["common.h"]
    assert re.search(r'__builtin_amdgcn_fence\(__ATOMIC_ACQ_REL, "wavefront"\)', found[0][1])
