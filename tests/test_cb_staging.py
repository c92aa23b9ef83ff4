"""The address arithmetic of the coherent kernels' FTPA staging loads
(csrc/cb_stage.hpp, which the kernels use) on the CPU: tests/cpp/test_staging.cpp
walks every load of a block's last tile for 4 to 128 antennas, whole blocks and
subsets at any place of a wider one, and reads the operands back."""
import os
import subprocess

EXE = os.path.join(os.path.dirname(__file__), "cpp", "test_staging")


def test_staged_loads_stay_in_the_block():
    src = EXE + ".cpp"
    if not os.path.exists(EXE):
        subprocess.run(["g++", "-O1", "-std=c++17", src, "-o", EXE], check=True, timeout=100)
    res = subprocess.run([EXE], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout[:2000]
