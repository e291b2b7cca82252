"""The dense path's mask (sentinel_amd/csrc/dense_mask.h) against the rule on positions, on the CPU (tests/cpp/test_dense_mask.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EXE = os.path.join(HERE, "cpp", "test_dense_mask")


def test_mask_is_the_rule_on_positions():
    if not os.path.exists(EXE):  # plain C++ (g++): no HIP compiler needed
        if shutil.which("make") is None or shutil.which(os.environ.get("CXX", "g++")) is None:
            pytest.skip("tests/cpp/test_dense_mask is not built and there is no make / C++ compiler to build it")
        subprocess.run(["make", "-C", os.path.join(HERE, "cpp"), EXE], check=True, capture_output=True, timeout=300)
    proc = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "dense mask ok" in proc.stdout
