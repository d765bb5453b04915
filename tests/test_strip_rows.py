"""The level-0 strips' addressing (imscript_amd/csrc/sp_strip.h) on the CPU:
no scalar offset exceeds its buffer, rows outside the image and the halo above
a tile are not touched, every pixel is stored once."""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT


@pytest.fixture(scope="module")
def strip_rows(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("strip") / "strip_rows")
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", exe,
                    os.path.join(ROOT, "tests", "cpu", "strip_rows.cpp")], check=True)
    return exe


# tile edges (108 x 44) and remainders, the smallest planes, odd widths
@pytest.mark.parametrize("size", ["2 2", "3 2", "2 3", "108 44", "107 43", "109 45", "216 88",
                                  "217 89", "330 133", "33 301", "1030 7"])
def test_rows_stay_in_their_buffers(strip_rows, size):
    p = subprocess.run([strip_rows, *size.split()], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr
    assert p.stdout.startswith("OK")
