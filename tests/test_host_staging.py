"""The pinned transfers (dg-bgk_amd/csrc/staging.hpp) on the CPU, on a
stand-in for the few HIP calls they make (tests/sanitize/hip_stub), under the
address and undefined-behaviour sanitizers and under the thread sanitizer."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SAN = os.path.join(ROOT, "tests", "sanitize")

pytestmark = pytest.mark.skipif(
    not os.path.isdir(SAN) or shutil.which("g++") is None,
    reason="sanitizer drivers or host compiler absent")


@pytest.mark.parametrize("san", ["address,undefined", "thread"])
def test_transfers_on_a_late_device(san, tmp_path):
    exe = str(tmp_path / "staging_check")
    subprocess.run(["g++", "-std=c++17", f"-fsanitize={san}", "-fno-sanitize-recover=all", "-g",
                    "-O1", "-pthread", "-I" + os.path.join(SAN, "hip_stub"),
                    "-I" + os.path.join(ROOT, "dg-bgk_amd", "csrc"),
                    os.path.join(SAN, "staging_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and "staging ok" in r.stdout, r.stderr[-3000:]
