"""The sizes that the packed convolutions accept (ml_framework_amd/csrc/packed_limits.h)
against the 32-bit offsets their kernels form: tests/cpp/test_packed_limits.cpp, on
the CPU, with planes of 20 million pixels and hundreds of thousands of channels."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_packed_limits(tmp_path):
    exe = tmp_path / "test_packed_limits"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    f"-I{os.path.join(ROOT, 'ml_framework_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "cpp", "test_packed_limits.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    assert "all checks passed" in out.stdout
