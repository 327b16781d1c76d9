"""The nested-dissection plan of the device factor (mdz_factor_plan.h) on the
host: factors built from the plan alone solve random matrices over staggered
lattices of odd sizes, with missing unknowns, every reach and periodic
walls."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_plan_factors_random_lattices(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    exe = str(tmp_path / "factor_plan_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", os.path.join(HERE, "factor_plan_check.cpp"), "-o", exe,
                    "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    print(r.stdout[-3000:])
    assert r.returncode == 0 and r.stdout.strip().endswith("0 failed")
