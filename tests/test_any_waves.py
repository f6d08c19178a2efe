"""The waves that the decode kernels for any number of columns run on (csrc/q8_gemv.h), compiled and run on
the host: every column has a lane, a tail only beside a whole number of waves a SIMD, and a tail's lanes
fit the workgroup for 8 rows of two matrices."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_waves_and_tails(tmp_path):
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "any_waves")
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "intel-phi-apl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "c", "any_waves.cpp"), "-o", exe], check=True, capture_output=True, timeout=300)
    lines = [tuple(map(int, s.split())) for s in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert len(lines) == 512
    for cols, waves, tail, lanes in lines:
        assert 1 <= waves <= 16 and 1024 * waves + 16 * tail >= cols and 1024 * (waves - 1) < cols, cols
        if tail:
            assert waves % 4 == 0, cols
            assert lanes >= tail and 16 * lanes <= 64 * waves, cols
    assert any(tail for *_, tail, _ in lines)
