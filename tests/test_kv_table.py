"""CPU: a cache's page table on the device holds what the host has mapped, whatever captures and their replays did before, and the
entries of a sequence that starts again are not uploaded where it gets the pages it had (csrc/kv_table.h, compiled for the host)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_entry_is_there_after_a_direct_call_and_a_restart_uploads_nothing(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "table")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "skainet_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "c", "kv_table.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 50000
