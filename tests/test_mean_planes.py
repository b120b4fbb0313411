"""Planes per sample of a launch of several jobs (CPU only): a host-only
program built with g++ from deep-mr_amd/csrc/tn_worklist.h."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_mean_planes(tmp_path):
    exe = tmp_path / "planes_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "deep-mr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "planes_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
