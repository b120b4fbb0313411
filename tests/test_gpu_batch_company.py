"""A plan's gridding does not depend on its company: in a batch whose partial
tiles together pass the fixed workspace (32 MiB) every plan's grid has the bits
of the plan's own launch."""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing
from tilenufft.batch import BatchedNUFFT

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("frames", [1, 3])
def test_batched_grids_equal_the_plans_own(frames):
    print(f"batch company frames={frames}", flush=True)
    rng = np.random.default_rng(7)
    coils = [32, 17, 32, 24]
    plans = [tilenufft.fft.plan_nufft(
        rng.normal(0, 9, (frames, 1, n // frames, 2)).clip(-32, 32).astype(np.float32), 64, 4, 1.5, device=DEV)
        for n in (150_000, 120_000, 180_000, 90_000)]
    b = BatchedNUFFT(plans, coils)
    b.kspace.copy_(testing.complex_normal(tuple(b.kspace.shape), seed=3))
    b.gridding(b.grid)
    floats = 0
    for k, (p, c) in enumerate(zip(plans, coils)):
        g = torch.empty((c, p.nframes, *p.os_shape), dtype=torch.complex64, device=DEV)
        p.interpolator.gridding(b.kspace_view(k).contiguous(), g, c)
        floats += p.interpolator._workspaces[c, 0]
        n = c * p.nframes
        start = b.grid_off[k] // int(np.prod(p.os_shape))
        assert torch.equal(torch.view_as_real(g.reshape(n, *p.os_shape)), torch.view_as_real(b.grid[start:start + n]))
    assert floats * 4 > 32 << 20
