"""Which plans a backward's two products get (plan.h): tests/cpp/test_pair_plans.cpp,
host code of the header, on the CPU."""
import os
import shutil
import subprocess

import pytest

from ml_framework_amd.build import CSRC, HIP_FLAGS, HIPCC

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which(HIPCC) is None and not os.path.exists(HIPCC), reason="hipcc not available")
def test_pair_plans(tmp_path):
    exe = tmp_path / "test_pair_plans"
    out = subprocess.run([HIPCC, *HIP_FLAGS, "-x", "hip", "--offload-host-only", f"-I{CSRC}",
                          os.path.join(ROOT, "tests", "cpp", "test_pair_plans.cpp"), "-o", str(exe)],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert "all checks passed" in out.stdout
