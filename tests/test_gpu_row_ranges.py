"""Whole 3D transforms leave out the grid cells that no footprint reaches: the
results (2D too, which transforms every cell) equal those of the separate stages over the full grid, bit for bit, in
workspaces that held NaN before."""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def coords(kind, shape, rng):
    nd = len(shape)
    n = np.asarray(shape[::-1], np.float32)
    if kind == "ball":
        v = rng.standard_normal((1, 700, nd))
        return (v / np.linalg.norm(v, axis=-1, keepdims=True) * rng.uniform(0, 0.49, (1, 700, 1)) * n).astype(np.float32)
    if kind == "corner":  # one quadrant at the edge: footprints wrap
        return (rng.uniform(0.4, 0.5, (1, 50, nd)) * n).astype(np.float32)
    if kind == "two":  # both ends of the axes only
        return (np.sign(rng.uniform(-1, 1, (1, 40, nd))) * rng.uniform(0.45, 0.49, (1, 40, nd)) * n).astype(np.float32)
    if kind == "lines":  # Cartesian y, a few rows
        c = rng.uniform(-0.5, 0.5, (1, 60, nd)).astype(np.float32) * n
        c[..., 1] = rng.choice([-5, 0, 3], (1, 60))
        return c
    frames = [coords(k, shape, rng)[:, :40] for k in ("ball", "corner", "two")]
    return np.stack(frames)  # ranges differ between the frames


@pytest.mark.parametrize("kind", ["ball", "corner", "two", "lines", "frames"])
@pytest.mark.parametrize("shape, osf, width", [
    ((20, 12), 2.0, 4),       # a tile across the middle of the rows (24 cells, tiles of 8)
    ((64, 64), 1.25, 3),
    ((128, 256), 2.0, 6),
    ((12, 20, 16), 2.0, 4),
    ((51, 16, 12), 2.0, 3),   # x of 24
    ((51, 13, 32), 1.25, 3),  # z of 64, y of 17, x of 40
])
def test_ranged_equals_full(kind, shape, osf, width):
    print(f"row ranges {kind} {shape}", flush=True)
    rng = np.random.default_rng(5)
    plan = tilenufft.fft.plan_nufft(coords(kind, shape, rng), shape, width, osf, device=DEV)
    nat, coils = plan.interpolator, 3
    if not nat.has_transform:
        pytest.skip("no stages")
    nf, nimg = nat.nframes, 3 * nat.nframes
    poison = torch.full((4 * nimg * int(np.prod(plan.os_shape)),), float("nan"), dtype=torch.complex64, device=DEV)

    x = testing.complex_normal((coils, nf, *shape), seed=1).to(DEV)
    grid = torch.zeros((nimg, *plan.os_shape), dtype=torch.complex64, device=DEV)
    nat.transform_forward(x, grid, nimg)
    ref = torch.empty((coils, nf, nat.npts), dtype=torch.complex64, device=DEV)
    nat.interp(grid, ref, coils)
    del grid, poison  # the transform's workspaces come from these
    assert torch.equal(nat.nufft_forward(x, coils), ref)

    y = testing.complex_normal((coils, nf, nat.npts), seed=2).to(DEV)
    grid = torch.empty((nimg, *plan.os_shape), dtype=torch.complex64, device=DEV)
    nat.gridding(y, grid, coils)
    ref = torch.empty((nimg, *shape), dtype=torch.complex64, device=DEV)
    nat.transform_adjoint(grid, ref, nimg)
    grid.fill_(float("nan"))
    del grid
    assert torch.equal(nat.nufft_adjoint(y, coils), ref)
