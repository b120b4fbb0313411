"""Launches of more workgroups than are resident at once (over 1024 items):
the staged interpolation takes its wide loads from a number of planes on, by
row below it, on either side against the gather kernel, which forms the same
sums in the same order, from grids 16-byte aligned and not.

Tolerance: sums of T = W^ndim products, each rounded once in both kernels.
"""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("shape, osf, frames, width, coils", [
    *[((64, 64), 2.0, 20, w, c) for w, c in ((3, 1), (4, 2), (4, 3), (5, 5), (5, 6), (6, 2), (6, 3), (7, 3))],
    *[((60, 63), 1.6667, 32, w, c) for w, c in ((4, 8), (6, 2), (6, 3))],  # odd rows
    *[((60, 60, 60), 2.0, 1, w, c) for w, c in ((4, 2), (4, 3), (5, 3))],
])
def test_large_launches_match_gather(shape, osf, frames, width, coils):
    print(f"staged planes {shape} W={width} osf={osf} frames={frames} coils={coils}", flush=True)
    rng = np.random.default_rng(width)
    npts = 400 if len(shape) == 2 else 20000
    coord = (rng.uniform(-0.5, 0.5, (frames, 1, npts, len(shape))) * np.asarray(shape[::-1])).astype(np.float32)
    staged, gather = (tilenufft.fft.plan_nufft(coord, list(shape), width, osf, device=DEV, interp_mode=m)
                      for m in (2, 1))
    tol = 2.0 * (width ** len(shape)) ** 0.5 * 2.0**-24
    n = coils * frames * int(np.prod(staged.os_shape))
    flat = testing.complex_normal((n + 1,), seed=7).to(DEV)
    for first in (0, 1):
        out = [torch.full((coils, frames, npts), float("nan"), dtype=torch.complex64, device=DEV) for _ in range(2)]
        for p, o in zip((staged, gather), out):
            p.interpolator.interp(flat[first:first + n], o, coils)
        assert float((out[0] - out[1]).norm() / out[1].norm()) < tol
