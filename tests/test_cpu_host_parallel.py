"""Loops over host data on threads (mdz_host_parallel.h) where a thread
cannot be started or a chunk throws: no call may end the process."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_no_thread_and_throwing_chunks(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    exe = str(tmp_path / "host_parallel_check")
    subprocess.run([cxx, "-O1", "-std=c++17", "-Wall", os.path.join(HERE, "host_parallel_check.cpp"), "-o", exe,
                    "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and r.stdout.strip().endswith("0 failed")
