"""FFT stages of grid lengths without a kernel of their own (factors up to 17,
chirp transforms) against the same steps in 64 bits: apodize, centred zero pad,
DFT, and back.

Tolerance: an axis passes twice through at most log2(1536) < 11 radix-2 levels
and six further products, each rounding by at most 2^-24 in the mean square.
"""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def plan_of(shape, osf):
    rng = np.random.default_rng(0)
    coord = rng.uniform(-0.5, 0.5, (3, 40, len(shape))).astype(np.float32) * np.asarray(shape[::-1], np.float32)
    return tilenufft.fft.plan_nufft(coord, shape, 3, osf, device=DEV)


@pytest.mark.parametrize("shape, osf, grid", [
    # factors up to 17: each radix, first, last and alone
    ((28, 28), 2.0, (56, 56)),
    ((3, 5), 1.25, (4, 7)),
    ((7, 27), 1.25, (9, 34)),
    ((64, 97), 1.25, (80, 122)),              # chirp along x (61), a kernel of its own along y
    ((80, 104), 1.25, (100, 130)),
    ((667, 28), (1.5, 1.25), (1001, 35)),     # 7 11 13
    ((231, 816), 1.25, (289, 1020)),          # 17 17; 3 4 5 17
    ((13, 31, 22), 1.25, (17, 39, 28)),
    ((12, 37, 61), 1.25, (15, 47, 77)),       # chirp along y between the others
    # chirp
    ((15, 18), 1.25, (19, 23)),               # the shortest
    ((53, 47), (1.43, 1.3), (76, 62)),        # N + G - 1 = 128 along y: the convolution holds nothing else
    ((54, 64), (1.4, 1.25), (76, 80)),        # one more: the next length
    ((512, 260), (2.0015, 1.25), (1025, 325)),  # N + G - 1 = 1536: the longest
    ((349, 251), 1.25, (437, 314)),           # 19 23; 157
    ((15, 37, 64), 1.25, (19, 47, 80)),
])
def test_stages_match_64_bits(shape, osf, grid):
    print(f"stages {shape} -> {grid}", flush=True)
    plan = plan_of(shape, osf)
    nat, nd, nimg = plan.interpolator, len(shape), 3
    assert tuple(plan.os_shape) == grid and nat.has_transform and not nat.has_fft
    tol = nd * (2 * 11 + 6) * 2.0**-24
    ax = tuple(range(1, nd + 1))
    apod = np.ones(shape)
    for d in range(nd):
        w = tilenufft._core.apodization(shape[d], plan.oversamp[d], plan.width[d], plan.beta[d])
        apod = apod * w.astype(np.float64).reshape([-1 if k == d else 1 for k in range(nd)])
    crop = (slice(None),) + tuple(slice(g // 2 - n // 2, g // 2 - n // 2 + n) for g, n in zip(grid, shape))

    x = testing.complex_normal((nimg, *shape), seed=1)
    pad = np.zeros((nimg, *grid), np.complex128)
    pad[crop] = x.numpy().astype(np.complex128) * apod
    ref = np.fft.fftn(np.fft.ifftshift(pad, axes=ax), axes=ax)
    out = torch.full((nimg, *grid), float("nan"), dtype=torch.complex64, device=DEV)
    nat.transform_forward(x.to(DEV), out, nimg)
    assert rel(out.cpu().numpy(), ref) < tol

    k = testing.complex_normal((nimg, *grid), seed=2)
    ref = np.fft.fftshift(np.fft.ifftn(k.numpy().astype(np.complex128), axes=ax), axes=ax)[crop] * apod
    img = torch.full((nimg, *shape), float("nan"), dtype=torch.complex64, device=DEV)
    nat.transform_adjoint(k.to(DEV), img, nimg)
    assert rel(img.cpu().numpy(), ref) < tol


def test_the_library_transforms_what_no_stage_does():
    n = 513  # grid 1026 = 2 27 19: N + G - 1 = 1538
    print("chirp fallback", flush=True)
    plan = plan_of((n, 64), 2.0)
    assert not plan.interpolator.has_transform
    x = testing.complex_normal((1, n, 64), seed=3).to(DEV)
    y = tilenufft.fft.apply_nufft(x, plan)
    k = testing.complex_normal(tuple(y.shape), seed=4).to(DEV)
    a = tilenufft.fft.apply_nufft_adj(k, plan) * float(np.prod(plan.os_shape))
    lhs, rhs = torch.vdot(k.flatten(), y.flatten()), torch.vdot(a.flatten(), x.flatten())
    assert abs(lhs - rhs) <= 1e-4 * abs(lhs)
