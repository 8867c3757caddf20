"""Workgroups of the row sweeps on rows of more than 512 cells
(deepgpr_amd/csrc/dgx_rows.h), and which of them the sweeps take. No GPU needed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_long_rows(tmp_path):
    exe = tmp_path / "row_threads_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    "-I" + os.path.join(ROOT, "deepgpr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "row_threads_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-3000:]
    assert "all checks passed" in res.stdout
