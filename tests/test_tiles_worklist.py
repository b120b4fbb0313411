"""Host-built work of the tile gridding (CPU only, no device): footprint
pieces, brick order and the deal over the XCDs (deep-mr_amd/csrc/tn_worklist.h),
checked by a host-only program built with g++ from that header."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_worklist_invariants(tmp_path):
    exe = tmp_path / "tiles_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "deep-mr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "tiles_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("ok "), out.stdout + out.stderr
