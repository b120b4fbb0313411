"""A fine grid_split on an automatic plan: the partial tiles are bounded by the
fixed gridding workspace (32 MiB), so allocation-free launches take the plan as
they do with the automatic split, and the results agree.

Tolerance: a cell's sum of n terms of size a is regrouped, n eps a: 1e-5 of the
largest cell.
"""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import _core, _lib, testing

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("ndim, samples, split, coils", [(2, 60_000, 4, 16), (3, 30_000, 8, 20), (2, 3_000, 64, 3)])
def test_static_gridding_takes_fine_splits(ndim, samples, split, coils):
    print(f"static gridding {ndim}D, {samples} samples, split {split}, {coils} coils", flush=True)
    n = 48 if ndim == 2 else 16
    coord = np.random.default_rng(1).normal(0.0, n / 10, (1, samples, ndim)).clip(-n / 2, n / 2).astype(np.float32)
    k = testing.complex_normal((coils, samples), seed=2).to(DEV)
    grids = []
    for sp in (split, 0):
        plan = tilenufft.fft.plan_nufft(coord, n, 4, 2.0, device=DEV, grid_split=sp)
        assert plan.interpolator.grid_mode_effective() == 4
        before = plan.interpolator.device_bytes()
        with torch.cuda.device(DEV):
            plan.interpolator.prepare(coils)
            assert plan.interpolator.device_bytes() - before < 48 << 20  # partial tiles and work list
            g = torch.full((coils, *plan.os_shape), float("nan"), dtype=torch.complex64, device=DEV)
            _lib.check(_lib.load().tn_grid_static(plan.interpolator.handle, _core.ptr(k), _core.ptr(g), coils, None,
                                                  _core.stream_ptr(DEV)), "tn_grid_static")
            own = torch.full_like(g, float("nan"))
            plan.interpolator.gridding(k, own, coils)
            torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(g), torch.view_as_real(own))
        grids.append(torch.view_as_real(g))
    assert float((grids[0] - grids[1]).abs().max()) <= 1e-5 * float(grids[1].abs().max())
