"""CPU: the workspace of the products follows the number of rows alone, whatever tiles the matrix takes, and tiles of 96 rows stay inside it
(csrc/gemm_rows.h, from which the host code takes the size and the kernel its blocks, compiled for the host)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_of_96_rows_read_inside_the_layout_of_64(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "rows")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "skainet_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "c", "gemm_rows.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 100000
