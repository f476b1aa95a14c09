"""The small-batch decode plan rule (velokv_plan.h), compiled for the host with g++ and swept over
skewed and uniform batches with true, unknown and wrong length sums."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_small_plan_bounds(tmp_path):
    exe = str(tmp_path / "small_plan_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "velo-core_amd", "csrc"), "-I",
                    os.path.join(ROOT, "include"), os.path.join(HERE, "csrc", "small_plan_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
