"""CPU: no load of the products of few rows depends on more of a buffer load's range check than its vector offset
(csrc/gemm_few_loads.h, from which the kernel takes its offsets, compiled for the host)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_load_is_inside_its_buffer_or_past_it_by_its_vector_offset(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "loads")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "skainet_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "c", "gemm_few_loads.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 100000
