"""Properties of the device code that no run shows reliably, read from its sources
and from the assembly that the compiler makes of them."""
import concurrent.futures
import glob
import os
import re
import subprocess

import pytest

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


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """The gfx950 assembly of each source, with the build's flags."""
    out = tmp_path_factory.mktemp("assembly")
    makefile = open(os.path.join(CSRC, "..", "Makefile")).read()
    hipcc = re.search(r"^HIPCC \?= (\S+)", makefile, re.M)[1]
    flags = re.search(r"^FLAGS := (.*?[^\\])$", makefile, re.M | re.S)[1].replace("\\\n", " ").split()
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")

    def compiled(path):
        to = str(out / (os.path.basename(path) + ".s"))
        subprocess.run([hipcc, *flags, "-S", "--offload-device-only", "-o", to, path], check=True, stderr=subprocess.DEVNULL)
        return os.path.basename(path), open(to).read()

    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        return dict(pool.map(compiled, [p for p in SOURCES if p.endswith(".hip")]))


def test_no_kernel_runs_out_of_registers(assembly):
    # Beyond 256 vector registers the compiler spills to accumulation registers, and
    # beyond those to memory, of which a kernel without matrix instructions needs none.
    for name, text in assembly.items():
        bodies = dict(re.findall(r"^(_Z\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, re.M | re.S))
        for accum, entry, spills in re.findall(r"- \.agpr_count: +(\d+)(.*?)\.vgpr_spill_count: +(\d+)", text, re.S):
            kernel = re.search(r"\.name: +(\w+)", entry)[1]
            assert int(spills) == 0, (name, kernel, int(spills))
            assert int(accum) == 0 or "v_mfma_" in bodies[kernel], (name, kernel, int(accum))


def test_no_value_is_copied_with_lanes_off(assembly):
    # A copy between registers at the head of the block where a branch's lanes join, before
    # the other lanes are turned back on, leaves those lanes an old value.
    copy = re.compile(r"(v_accvgpr_(write|mov|read)\S*|v_mov_b(32|64)\S*) [av]\S+, [av]\d*\S*$")
    for name, text in assembly.items():
        head = None  # vector and memory instructions since the block's label, or None past its head
        for line in text.splitlines():
            op = line.strip()
            if line.startswith(".LBB"):
                head = []
            elif head is None or not op or op[0] in ";.":
                continue
            elif op.startswith("s_or_b64 exec, exec"):
                assert not head or not all(copy.match(x) for x in head), (name, head)
                head = None
            elif op.startswith(("s_cbranch", "s_branch")) or "saveexec" in op:
                head = None
            elif op.startswith(("v_", "global_", "ds_")) and not op.startswith(("v_readlane", "v_writelane", "v_readfirst")):
                head.append(op)
