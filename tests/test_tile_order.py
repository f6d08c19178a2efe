"""The long prompts' tiles (csrc/q8_tile.hip) wait for a stage of limbs by counting the loads issued after
it: a step's weight loads must follow its last stage load. Read from the compiled kernels' assembly (no
GPU): in every step the order holds, and a scheduling barrier stands between the two kinds, so that no
compiler's schedule may mix them."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "intel-phi-apl_amd")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("tile") / "q8_tile.s")
    make = open(os.path.join(LIB, "Makefile")).read()
    flags = re.search(r"^HIPFLAGS = (.*)$", make, re.M).group(1).replace("$(ARCH)", "gfx950").split()
    subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", "csrc/q8_tile.hip", "-o", out], cwd=LIB, check=True, capture_output=True, timeout=300)
    return open(out).read()


def steps(body):
    """The body between barriers, each as a string: S a stage load (to LDS), W a weight or scale load, | a
    scheduling barrier, and its last vmcnt wait."""
    for part in re.split(r"^\s*s_barrier\s*$", body, flags=re.M):
        marks, wait = "", None
        for line in part.splitlines():
            line = line.strip()
            if line.startswith("buffer_load") and line.endswith(" lds"):
                marks += "S"
            elif line.startswith("global_load"):
                marks += "W"
            elif "sched_barrier" in line:
                marks += "|"
            elif line.startswith("s_waitcnt") and "vmcnt" in line:
                wait = int(re.search(r"vmcnt\((\d+)\)", line).group(1))
        yield marks, wait


def test_stage_loads_come_before_the_weights(assembly):
    kernels = re.findall(r"^_Z9gemm_tileILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E\S*:.*?\n(.*?)s_endpgm", assembly, re.S | re.M)
    assert len(kernels) == 10
    for *c, body in kernels:
        mt, rt, nw, np, nb, kg = map(int, c)
        si, tr = (mt * 6 + nw - 1) // nw, np * rt
        found = list(steps(body))
        # the prologue: nb - 1 stages, each with the weights of its pair after it (nb == 2: one pair's before)
        assert found[0][0].replace("|", "") == ("W" * 2 * tr if nb == 2 else "") + ("S" * si + "W" * 2 * tr) * (nb - 1), c
        whole = [m for m, _ in found[1:] if "S" in m]
        assert len(whole) == (4 if nb == 4 else 6), c  # the unrolled steps
        for marks in whole:
            loads = marks.replace("|", "")
            assert loads.startswith("S" * si + "W" * 2 * tr) and "S" not in loads[si:], (c, marks)
            assert "|" in marks[marks.rindex("S"):marks.index("W")], (c, marks)
        for _, wait in found[:len(whole)]:
            assert wait is not None and wait <= (nb - 2) * (si + 2 * tr) + 2 * tr, (c, wait)
