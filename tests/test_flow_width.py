"""The launch width of the sweeps without barriers (scisim_amd/csrc/scx_tune.h, host code):
tests/cpp/flow_width_tests.cpp."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_grid_fits_the_device(tmp_path):
    out = str(tmp_path / "flow_width_tests")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "scisim_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "flow_width_tests.cpp"), "-o", out], check=True)
    p = subprocess.run([out], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stderr
    assert "flow width tests passed" in p.stdout
