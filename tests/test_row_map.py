"""The block map of the row sweeps (deepgpr_amd/csrc/dgx_rows.h), checked on
the host over random grids, CPML widths and orders. No GPU needed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_row_map_covers_every_cell_once(tmp_path):
    exe = tmp_path / "row_map_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    "-I" + os.path.join(ROOT, "deepgpr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "row_map_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-3000:]
    assert "all checks passed" in res.stdout
