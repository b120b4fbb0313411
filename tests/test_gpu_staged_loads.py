"""The staged interpolation's region loads (pairs of cells, single cells, row by
row) against the gather kernel, which forms the same sums in the same order.

Tolerance: sums of T = W^ndim products, each rounded once in both kernels.
"""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def plans(shape, width, osf, **kw):
    rng = np.random.default_rng(width)
    coord = rng.uniform(-0.5, 0.5, (2, 900, len(shape))).astype(np.float32) * np.asarray(shape[::-1], np.float32)
    return [tilenufft.fft.plan_nufft(coord, shape, width, osf, device=DEV, interp_mode=m, **kw) for m in (2, 1)]


@pytest.mark.parametrize("shape, width, osf, coils, kw", [
    *[((40, 50), w, 2.0, 9, {}) for w in range(1, 9)],          # pairs; row by row from 7 taps on
    *[((31, 45), w, 1.0 + 2 / 3, 3, {}) for w in (3, 4, 6)],    # odd rows: single cells
    ((10, 9), 4, 1.25, 2, {}),                                  # one tile wider than the grid's rows
    ((40, 50), 4, 2.0, 9, {"interp_chunk": 3}),
    ((40, 50), 4, 2.0, 9, {"interp_chunk": 9}),                 # more coils than a chunk of the loads
    ((40, 50), 4, 2.0, 9, {"itile": (24, 40)}),                 # a larger region
    ((40, 50), 4, 2.0, 9, {"itile": (8, 7)}),                   # tiles from odd cells on
    *[((14, 18, 20), w, 2.0, 3, {}) for w in range(1, 7)],      # pairs; row by row from 6 taps on
    ((13, 18, 21), 4, 1.6667, 5, {}),                           # odd rows: row by row
])
def test_staged_loads_match_gather(shape, width, osf, coils, kw):
    print(f"staged loads {shape} W={width} osf={osf} coils={coils} {kw}", flush=True)
    staged, gather = plans(shape, width, osf, **kw)
    tol = 2.0 * (width ** len(shape)) ** 0.5 * 2.0**-24
    n = coils * int(np.prod(staged.os_shape))
    flat = testing.complex_normal((n + 1,), seed=7).to(DEV)
    for first in (0, 1):  # 16-byte aligned, and not
        grid = flat[first:first + n]
        out = [torch.full((coils, 1800), float("nan"), dtype=torch.complex64, device=DEV) for _ in range(2)]
        for p, o in zip((staged, gather), out):
            p.interpolator.interp(grid, o, coils)
        assert float((out[0] - out[1]).norm() / out[1].norm()) < tol
