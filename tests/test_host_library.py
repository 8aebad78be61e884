"""The library's host code checked from the inside, on the CPU: tests/sanitize/host_library.cpp takes in
tmk_api.hip, is built host only with AddressSanitizer and UndefinedBehaviorSanitizer and runs against the
host-memory stand-in of the HIP runtime, so that the tables a launch would read are plain host memory.

registers: of every face that a hierarchy's flux registers read, exactly one workgroup of the level's
launch stores the flux, with regions that end 3 coarse cells from the fault and from the other edges,
where strips and boundary pieces meet.
scratch_limit: the allocation-free drop-in call takes and refuses the boxes it always did, by bytes near
its limit.
strip_lists: the strips and boundary pieces of every FP64 box that call takes fit its list.
stages: the pinned buffers of downloads and drop-in calls: bounded for each device, never pinned and freed
over and over, by ten devices or forty readers, and none needed.
upload_staging: an upload takes no more device memory than the box's planes in the level's type, small
boxes aside.
reader_threads: a download whose threads cannot be started for want of host memory carries its pieces on
by itself.
strip_heights: the height a level reports is the one its launches take, and levels that report the same
share launches.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitize")


@pytest.fixture(scope="module")
def driver():
    if not (os.path.exists("/opt/rocm/bin/hipcc") and os.path.exists("/opt/rocm/llvm/bin/clang++") and shutil.which("make")):
        pytest.skip("needs ROCm's hipcc and clang++ and make")
    b = subprocess.run(["make", "-j4", "_build/host_library"], cwd=HERE, capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stdout[-4000:] + b.stderr[-4000:]
    return os.path.join(HERE, "_build", "host_library")


@pytest.mark.parametrize("check", ["registers", "scratch_limit", "strip_lists", "stages", "upload_staging", "reader_threads", "strip_heights"])
def test_host_library(driver, check):
    r = subprocess.run([driver, check], cwd=HERE, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and check + " ok" in r.stdout, r.stdout[-4000:] + r.stderr[-8000:]
