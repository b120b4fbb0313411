"""Many steps of one wave (sixteen entries each, handed from lane to lane
through its LDS): every sample in one tile, unsplit, against the gridding
matrix, and twice (same bits).

Tolerance: the matrix sums its long rows in parts, so a cell's n terms are
grouped differently: each side is within n eps of the sum of their magnitudes
(the gridding of the samples' magnitudes, the weights are positive).
"""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("ndim, width", [(2, 4), (2, 6), (3, 4), (3, 5)])
@pytest.mark.parametrize("coils", [1, 9, 20, 32])
def test_long_tiles_equal_the_matrix(ndim, width, coils):
    print(f"long tiles {ndim}D W={width} coils={coils}", flush=True)
    rng = np.random.default_rng(coils)
    coord = rng.uniform(1.6, 2.9, (1, 1003, ndim)).astype(np.float32)
    k = testing.complex_normal((coils, 1, 1003), seed=3).to(DEV)
    grids = []
    for mode, y in ((0, k), (3, k), (0, k), (3, torch.complex(k.real.abs(), k.imag.abs()))):
        p = tilenufft.fft.plan_nufft(coord, 16, width, 2.0, device=DEV, grid_mode=mode, grid_split=-1)
        assert p.interpolator.grid_mode_effective() == (4 if mode == 0 else 3)
        g = torch.full((coils, 1, *p.os_shape), float("nan"), dtype=torch.complex64, device=DEV)
        p.interpolator.gridding(y, g, coils)
        grids.append(torch.view_as_real(g))
    assert torch.equal(grids[0], grids[2])
    assert ((grids[0] - grids[1]).abs() <= 2 * 1003 * 2.0**-24 * grids[3]).all()
