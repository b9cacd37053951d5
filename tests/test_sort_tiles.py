"""Tile sizes of the radix passes, on the host (tests/cpp/sort_tiles_test.cpp,
compiled with hipcc; it makes no HIP calls)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "dendro4_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not found")
def test_tiles_match_the_kernels(tmp_path):
    exe = tmp_path / "sort_tiles_test"
    cmd = [HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "-I", CSRC,
           os.path.join(ROOT, "tests", "cpp", "sort_tiles_test.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "0 failures" in r.stdout, r.stdout + r.stderr
