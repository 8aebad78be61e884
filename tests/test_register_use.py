"""The FP64 interior kernels that carry both sides of a cell in one thread are held to 128 vector registers
(two workgroups on a CU); what does not fit is spilled to memory on every cell.  Compiled for gfx950 (no
GPU needed), a few registers at most may be: 52 spilled made a step half as long again.
"""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = "/opt/rocm/bin/hipcc"
SOURCE = """#include <hip/hip_runtime.h>
#include "tetemoko_hip.h"
#include "tmk_kernels.hpp"
#include "tmk_interior.hpp"
namespace tmk {
template __global__ void k_godunov_interior<double, 2, 32, 16, PK_PPM_PRIM>(const KArgs<double>);
template __global__ void k_godunov_interior<double, 2, 64, 8, PK_PPM_PRIM>(const KArgs<double>);
template __global__ void k_godunov_interior<double, 2, 64, 16, PK_PPM_PRIM>(const KArgs<double>);
template __global__ void k_godunov_interior<double, 2, 32, 32, PK_PPM_PRIM>(const KArgs<double>);
}
"""


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="needs hipcc")
def test_both_sides_in_one_thread_stay_in_registers(tmp_path):
    src = tmp_path / "k.hip"
    src.write_text(SOURCE)
    r = subprocess.run([HIPCC, "-O3", "--offload-arch=gfx950", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-ffp-contract=off", "--cuda-device-only", "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(ROOT, "tetemoko_amd", "csrc"), "-Rpass-analysis=kernel-resource-usage",
                        "-c", str(src), "-o", str(tmp_path / "k.o")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    use = re.findall(r"Function Name: \S*k_godunov_interiorIdLi2ELi(\d+)ELi(\d+)E\S*.*?VGPRs Spill: (\d+)", r.stderr, re.S)
    assert len(use) == 4
    for bx, by, spill in use:
        assert int(spill) <= 10, (bx, by, spill)
