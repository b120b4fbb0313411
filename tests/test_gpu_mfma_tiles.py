"""GPU parity of the automatic tile gridding (matrix cores) beyond what
grid_mode 4 accepts: 2D plans, odd and tiny grids, widths up to 6, Cartesian
axes, every block count, and the coil-minor copy, against the gridding matrix.

Without splits (grid_split -1) both variants add a cell's terms (wz wy) wx *
scaled sample in ascending sample order with one rounding each, so the grids
are the same bits. With the default splits a cell's sum is regrouped: n terms of
size a differ by at most n eps a, bounded here by 1e-5 of the largest cell. A
sample that is not finite reaches the cells of its footprint only, as in the
matrix.
"""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def grids(coord, shape, width, osf, coils, split, k=None):
    """The gridded k-space of the automatic (tile) plan and of the matrix plan."""
    out = []
    for mode in (0, 3):
        p = tilenufft.fft.plan_nufft(coord, shape, width, osf, device=DEV, grid_mode=mode, grid_split=split)
        assert p.interpolator.grid_mode_effective() == (4 if mode == 0 else 3)
        if k is None:
            k = testing.complex_normal((coils, p.nframes, p.npts), seed=3).to(DEV)
        g = torch.full((coils, p.nframes, *p.os_shape), float("nan"), dtype=torch.complex64, device=DEV)
        p.interpolator.gridding(k, g, coils, torch.linspace(0.5, 1.5, p.nframes * p.npts, device=DEV))
        torch.cuda.synchronize()
        out.append(torch.view_as_real(g))
    return out


CASES = [
    # (shape, width, osf, coils, frames, samples)
    ((24, 24), 4, 2.0, 1, 1, 500),      # one coil
    ((25, 37), 4, 1.25, 3, 2, 400),     # ragged tiles, frames
    ((30, 22), 3, 1.5, 8, 1, 700),
    ((27, 27), 5, 1.25, 9, 1, 300),     # 8-tap records, two blocks
    ((20, 33), 6, 1.5, 17, 1, 300),     # three blocks
    ((6, 5), 4, 1.25, 2, 1, 60),        # grids shorter than a tile and a footprint: both pieces in one tile
    ((7, 40), 2, 1.25, 33, 1, 200),     # two chunks of coils
    ((40,), 4, 1.25, 4, 2, 90),         # 1D: one grid row
    ((13, 17, 11), 4, 1.25, 5, 1, 900),  # ragged 3D
    ((9, 10, 12), 6, 1.5, 2, 1, 300),
    ((3, 16, 16), 4, 1.5, 8, 1, 300),   # a grid of one ragged z tile
]


@pytest.mark.parametrize("shape, width, osf, coils, frames, samples", CASES)
def test_tiles_equal_matrix_bitwise_without_splits(shape, width, osf, coils, frames, samples):
    print(f"tiles {shape} W={width} osf={osf} coils={coils} frames={frames}", flush=True)
    rng = np.random.default_rng(7)
    lim = np.array(shape[::-1]) / 2
    coord = rng.uniform(-lim, lim, (frames, 1, samples, len(shape))).astype(np.float32)
    a, b = grids(coord, list(shape), width, osf, coils, -1)
    assert torch.equal(a, b)


def test_tiles_with_a_cartesian_axis():
    """x on the grid (width 1), y off it: two frames whose lines differ."""
    ky, kx = np.meshgrid(np.linspace(-15.5, 15.5, 30), np.arange(-16, 16), indexing="ij")
    coord = np.stack([np.stack([kx, ky + s], -1) for s in (0.2, -0.3)]).astype(np.float32)
    a, b = grids(coord, [32, 32], 4, 1.25, 3, -1)
    assert torch.equal(a, b)


@pytest.mark.parametrize("ndim, split", [(2, 0), (2, 48), (3, 0), (3, 40)])
def test_hot_tiles_shared_and_split(ndim, split):
    """A dense centre: tiles shared by a workgroup's four waves (more than 96
    samples, or split / 4) and tiles split over workgroups, twice (bitwise)."""
    rng = np.random.default_rng(11)
    n = 20
    coord = np.concatenate([rng.uniform(-n / 2, n / 2, (1, 600, ndim)), rng.normal(0, 0.4, (1, 3000, ndim))],
                           1).astype(np.float32)
    a, b = grids(coord, n, 4, 2.0, 10, split)
    assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())
    a2, _ = grids(coord, n, 4, 2.0, 10, split)
    assert torch.equal(a, a2)


def test_large_tables_read_a_copy():
    """More than 48 MiB of samples (11 coils x 600,000): the coil-minor copy,
    a partial record in the second chunk of eight."""
    coord = np.random.default_rng(12).uniform(-20, 20, (1, 600_000, 2)).astype(np.float32)
    a, b = grids(coord, 40, 4, 2.0, 11, -1)
    assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


@pytest.mark.parametrize("shape", [(24, 24), (12, 12, 12)])
def test_values_that_are_not_finite_stay_in_their_footprints(shape):
    rng = np.random.default_rng(13)
    n = shape[0]
    coord = rng.uniform(-n / 2, n / 2, (1, 200, len(shape))).astype(np.float32)
    k = testing.complex_normal((3, 1, 200), seed=4).to(DEV)
    k[0, 0, 5] = float("nan")
    k[1, 0, 17] = complex(float("inf"), 1.0)
    a, b = grids(coord, list(shape), 4, 2.0, 3, -1, k)
    assert torch.equal(torch.isfinite(a), torch.isfinite(b)) and not torch.isfinite(a).all()
    fin = torch.isfinite(a)
    assert torch.equal(a[fin], b[fin])
    assert torch.isnan(a[0][~fin[0]]).all() and fin[2].all()
    # coil 1: positive weights times a real part of +inf stay +inf (the matrix
    # kernel's masked loads can turn them into NaN), the imaginary part is finite
    re, im = a[1][..., 0], a[1][..., 1]
    assert (re[~torch.isfinite(re)] == float("inf")).all() and torch.isfinite(im).all()
