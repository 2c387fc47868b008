"""Which kernels a call runs on (ml_framework_amd/csrc/conv_routes.h, gemm_routes.h)
against tables of calls timed on both sides on one MI355X (tests/golden/*_routes.csv):
tests/cpp/test_routes.cpp, on the CPU. A rule that sends a timed call to the clearly
slower side shows here."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_routes(tmp_path):
    exe = tmp_path / "test_routes"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    f"-I{os.path.join(ROOT, 'ml_framework_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "cpp", "test_routes.cpp"), "-o", str(exe)], check=True)
    tables = [os.path.join(ROOT, "tests", "golden", f"{n}_routes.csv") for n in ("conv", "gemm")]
    out = subprocess.run([str(exe), *tables], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "all checks passed" in out.stdout
