"""The brick lists' sizes, on the CPU (tests/host/list_bounds.hip): the chunk
limit keeps every list offset within an int, and no section hits more bricks
than its buffer share."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not available")
def test_list_bounds(tmp_path):
    exe = str(tmp_path / "list_bounds")
    subprocess.check_call([HIPCC, "-std=c++17", "-O2", "--offload-arch=gfx950", "-ffp-contract=off",
                           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                           "-I", os.path.join(ROOT, "spider_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                           "-o", exe, os.path.join(HERE, "host", "list_bounds.hip")],
                          stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr
    assert "list bound checks passed" in p.stdout, p.stdout + p.stderr
