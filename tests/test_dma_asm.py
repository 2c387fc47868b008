"""The LDS-DMA load of half_tile.h is written in asm that sets M0: the compiler
has to know it, or a value it keeps in M0 itself could be taken for the old one.
Compiles one load for gfx950 on the CPU and reads the asm's constraints from the
compiler's intermediate form."""
import os
import re
import shutil
import subprocess

import pytest

from ml_framework_amd.build import CSRC, HIP_FLAGS, HIPCC

SOURCE = """
#include "half_tile.h"
__global__ void one_load(const seera::half_t* in, float* out) {
    __shared__ seera::half_t lds[512];
    seera::dma16(seera::make_dma_rsrc(in, 1024), lds, threadIdx.x * 16, 0);
    seera::wait_vm<0>();
    __syncthreads();
    out[threadIdx.x] = (float)lds[threadIdx.x];
}
"""


@pytest.mark.skipif(shutil.which(HIPCC) is None and not os.path.exists(HIPCC), reason="hipcc not available")
def test_dma_load_declares_m0(tmp_path):
    src = tmp_path / "one_load.hip"
    src.write_text(SOURCE)
    ir = tmp_path / "one_load.ll"
    out = subprocess.run([HIPCC, *HIP_FLAGS, f"-I{CSRC}", "--cuda-device-only", "-emit-llvm", "-S", str(src), "-o", str(ir)],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    constraints = re.findall(r'asm sideeffect "[^"]*buffer_load_dwordx4[^"]*lds", "([^"]*)"', ir.read_text())
    assert constraints and all("~{m0}" in c and "~{memory}" in c for c in constraints), constraints
