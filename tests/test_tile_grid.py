"""How the persistent grids share tiles out over XCDs and workgroups (sentinel_amd/csrc/grid_plan.h), run on the CPU: the compiled
check (tests/cpp/test_tile_grid.cpp) walks the grids as the kernels do, every tile has to be taken exactly once."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EXE = os.path.join(HERE, "cpp", "test_tile_grid")


def test_every_tile_is_taken_once():
    if not os.path.exists(EXE):  # plain C++ (g++): no HIP compiler needed
        if shutil.which("make") is None or shutil.which(os.environ.get("CXX", "g++")) is None:
            pytest.skip("tests/cpp/test_tile_grid is not built and there is no make / C++ compiler to build it")
        subprocess.run(["make", "-C", os.path.join(HERE, "cpp"), EXE], check=True, capture_output=True, timeout=300)
    proc = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "tile grid ok" in proc.stdout
