"""The Toeplitz operator's fused stages against the same steps in 64 bits.

Tolerance: a forward and an inverse transform per axis, each within the bound
of the FFT stages (twice 11 radix-2 levels and six products, 2^-24 each).
"""

import copy
import pickle

import pytest
import torch

from tilenufft import testing
from tilenufft.fft.toeplitz import GramMatrix, apply_nufft_selfadj

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(x, value, grid):
    nd = len(grid)
    ax = tuple(range(-nd, 0))
    x = x.to(torch.complex128)
    sl = (Ellipsis,) + tuple(slice(g // 2 - n // 2, g // 2 - n // 2 + n) for g, n in zip(grid, x.shape[-nd:]))
    big = torch.zeros((*x.shape[:-nd], *grid), dtype=torch.complex128, device=x.device)
    big[sl] = x
    return torch.fft.ifftn(value.to(torch.complex128) * torch.fft.fftn(big, dim=ax), dim=ax)[sl]


def check(y, x, value, grid):
    ref = reference(x, value, grid)
    assert y.shape == ref.shape and y.dtype == torch.complex64 and y.is_contiguous()
    assert float((y - ref).norm() / ref.norm()) < 2 * len(grid) * (2 * 11 + 6) * 2.0**-24


@pytest.mark.parametrize("lead, klead, shape, grid", [
    ((3,), (), (64, 40), (128, 80)),              # kernels of their own length
    ((5,), (), (33, 51), (66, 102)),              # factors up to 17
    ((2,), (), (23, 29), (46, 58)),               # chirp
    ((), (), (1, 1), (2, 2)),                     # the smallest
    ((2, 3), (3,), (20, 28), (40, 56)),           # one kernel per contrast: rows repeat inside a wave
    ((7,), (), (128, 257), (256, 514)),           # 514 = 2 257
    ((2,), (), (31, 64), (31, 128)),              # a Cartesian axis: no padding
    ((2, 2), (2,), (5, 12, 19), (10, 24, 38)),
    ((3,), (), (16, 64, 33), (32, 128, 66)),
    ((1,), (), (600, 16), (1200, 32)),            # N + G - 1 = 1799: the library transforms
    ((2,), (), (24, 24), (20, 24)),               # cropped to the grid: the library transforms
])
def test_convolution_matches_64_bits(lead, klead, shape, grid):
    print(f"convolve {lead} {klead} {shape} {grid}", flush=True)
    value = testing.complex_normal((*klead, *grid), seed=1).to(DEV)
    kern = GramMatrix(value, grid, len(grid), DEV, False)
    x = testing.complex_normal((*lead, *shape), seed=2).to(DEV)
    if any(n > g for n, g in zip(shape, grid)):
        assert kern.stages(shape, torch.device(DEV)) is None
        assert apply_nufft_selfadj(x, kern).shape == x.shape
        return
    check(apply_nufft_selfadj(x, kern), x, value, grid)


def test_forms_of_image_and_kernel():
    print("convolve forms", flush=True)
    grid, n = (48, 60), (24, 30)
    value = testing.complex_normal(grid, seed=3).to(DEV)
    kern = GramMatrix(value, grid, 2, DEV, False)
    x = testing.complex_normal((4, *n), seed=4).to(DEV)
    check(apply_nufft_selfadj(x.real.contiguous(), kern), x.real, value, grid)  # real images
    check(apply_nufft_selfadj(x.conj(), kern), x.conj().resolve_conj(), value, grid)
    t = x.transpose(-1, -2).contiguous().transpose(-1, -2)  # strided
    check(apply_nufft_selfadj(t, kern), x, value, grid)
    small = x[..., 3:, 5:28]  # another size through the same kernel, at an odd offset in memory
    check(apply_nufft_selfadj(small, kern), small, value, grid)
    kern.value = value.T.contiguous().T * 2.0  # the value in use is the value asked for
    check(apply_nufft_selfadj(x, kern), x, 2.0 * value, grid)
    for other in (copy.deepcopy(kern), pickle.loads(pickle.dumps(kern))):
        check(apply_nufft_selfadj(x, other), x, 2.0 * value, grid)


def test_capture_with_and_without_stages_built():
    print("convolve capture", flush=True)
    grid, n = (64, 64), (32, 32)
    value = testing.complex_normal(grid, seed=5).to(DEV)
    x = testing.complex_normal((2, *n), seed=6).to(DEV)
    kern = GramMatrix(value, grid, 2, DEV, False)
    apply_nufft_selfadj(x, kern)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        apply_nufft_selfadj(x, kern)
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        y = apply_nufft_selfadj(x, kern)
    for k in range(3):
        x.copy_(testing.complex_normal((2, *n), seed=7 + k))
        graph.replay()
        assert torch.equal(y, apply_nufft_selfadj(x, kern))
