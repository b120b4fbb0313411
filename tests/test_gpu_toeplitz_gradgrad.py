"""The Toeplitz operator differentiated twice: its backward, when a graph of it
is asked for, is made of torch's calls, which autograd records.

Tolerance: two applications, each within the bound of the FFT stages (twice 11
radix-2 levels and six products, 2^-24 each, per axis) on either side.
"""

import pytest
import torch

from tilenufft import testing
from tilenufft.fft.toeplitz import GramMatrix, apply_nufft_selfadj

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("shape, grid", [((24, 40), (48, 80)), ((9, 12, 10), (18, 24, 20))])
def test_second_derivatives(shape, grid):
    print(f"toeplitz second derivatives {shape} {grid}", flush=True)
    value = testing.complex_normal(grid, seed=1).real.abs().to(torch.complex64).to(DEV)  # self-adjoint
    kern = GramMatrix(value, grid, len(grid), DEV, False)
    ax = tuple(range(-len(grid), 0))
    sl = (Ellipsis,) + tuple(slice(g // 2 - n // 2, g // 2 - n // 2 + n) for g, n in zip(grid, shape))

    def reference(x):
        big = torch.nn.functional.pad(torch.view_as_real(x).movedim(-1, 0), [
            p for g, n in zip(grid[::-1], shape[::-1]) for p in (g // 2 - n // 2, g - n - (g // 2 - n // 2))])
        big = torch.complex(big[0], big[1])
        return torch.fft.ifftn(value.to(torch.complex128) * torch.fft.fftn(big, dim=ax), dim=ax)[sl]

    def second(op, x):
        x = x.clone().requires_grad_()
        (g,) = torch.autograd.grad((op(x).abs() ** 2).sum(), x, create_graph=True)
        assert g.requires_grad
        (h,) = torch.autograd.grad((g.real ** 2).sum(), x)
        return h

    x = testing.complex_normal((2, *shape), seed=2).to(DEV)
    got, ref = second(lambda t: apply_nufft_selfadj(t, kern), x), second(reference, x.to(torch.complex128))
    assert float((got - ref).norm() / ref.norm()) < 4 * 2 * len(grid) * (2 * 11 + 6) * 2.0**-24
