"""The kernels' plans and grids (plain C++ headers under bus-fill_amd/csrc)
checked on the CPU: tests/plan_check.cpp compiled with g++."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("plans") / "plan_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                    "-I", os.path.join(ROOT, "bus-fill_amd", "csrc"),
                    os.path.join(ROOT, "tests", "plan_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("part", ["dequant", "block_grid", "block_choice", "tile_grid"])
def test_plans(checker, part):
    r = subprocess.run([checker, part], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
