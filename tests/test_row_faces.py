"""Which CPML faces the row sweeps take (deepgpr_amd/csrc/dgx_rows.h): none
that a thread on the other half of the axis would have to look at. Brute force
on the host; no GPU needed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_row_sweeps_look_at_the_only_face_in_reach(tmp_path):
    exe = tmp_path / "row_face_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    "-I" + os.path.join(ROOT, "deepgpr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "row_face_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-3000:]
    assert "all checks passed" in res.stdout
