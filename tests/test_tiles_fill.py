"""Tiles without samples are zeroed in runs (tile gridding): the runs on the
CPU (deep-mr_amd/csrc/tn_worklist.h), and sparse trajectories on the GPU, whose
grids equal the gridding matrix's bit for bit in a workspace that held NaN, and
whose whole adjoints (which leave out cells that nothing reads) do too."""

import os
import subprocess

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda:0"


def test_runs_of_empty_tiles(tmp_path):
    exe = tmp_path / "fill_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "deep-mr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "fill_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("ok "), out.stdout + out.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("shape, osf, coils, frames, samples", [
    ((150, 67), 1.5, 1, 1, 3),        # rows of more than one run, an odd grid
    ((64, 96), 2.0, 9, 2, 20),
    ((5, 300), 1.25, 33, 1, 4),       # two chunks of coils
    ((21, 37, 75), 1.25, 9, 1, 12),   # ragged 3D, odd rows
    ((32, 32, 64), 2.0, 8, 1, 40),    # stages that skip unread cells
    ((16, 20, 48), 2.0, 2, 2, 1),
    ((12, 12, 12), 2.0, 3, 1, 0),     # no samples at all
])
def test_sparse_grids_equal_the_matrix(shape, osf, coils, frames, samples):
    print(f"sparse tiles {shape} osf={osf} coils={coils} frames={frames} samples={samples}", flush=True)
    rng = np.random.default_rng(5)
    lim = np.array(shape[::-1]) / 2
    coord = rng.uniform(-lim, lim, (frames, 1, samples, len(shape))).astype(np.float32)
    k = testing.complex_normal((coils, frames, 1, samples), seed=3).to(DEV)
    grids, images = [], []
    for mode in (0, 3):
        p = tilenufft.fft.plan_nufft(coord, list(shape), 4, osf, device=DEV, grid_mode=mode, grid_split=-1)
        assert p.interpolator.grid_mode_effective() == (4 if mode == 0 else 3)
        g = torch.full((coils, frames, *p.os_shape), float("nan"), dtype=torch.complex64, device=DEV)
        p.interpolator.gridding(k.reshape(coils, frames, samples), g, coils)
        grids.append(torch.view_as_real(g))
        images.append(torch.view_as_real(tilenufft.fft.apply_nufft_adj(k if frames > 1 else k[:, 0], p)))
    assert torch.equal(*grids) and torch.equal(*images)
