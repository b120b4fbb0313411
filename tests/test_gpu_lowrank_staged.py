"""The staged low-rank interpolation against the gathering one (interp_mode 1),
which the oracle tests pin: the same sums, in FP32 with other contractions, so
within 1e-6 relative L2. Coefficient counts that end inside and across the
planes loaded together, odd plane counts, a density weight, a dense centre
(tiles of several segments), 2D and 3D."""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("ndim, n, coils, nframes, ncoeff", [
    (2, 32, 1, 3, 1), (2, 32, 3, 7, 3), (2, 45, 5, 9, 5), (2, 32, 2, 12, 9), (3, 14, 3, 5, 4), (3, 12, 1, 4, 3),
])
def test_staged_equals_gather(ndim, n, coils, nframes, ncoeff):
    print(f"low rank {ndim}D n={n} coils={coils} frames={nframes} coeff={ncoeff}", flush=True)
    rng = np.random.default_rng(ncoeff)
    coord = rng.uniform(-n / 2, n / 2, (nframes, 1, 301, ndim)).astype(np.float32)
    coord[:, :, :200] *= 0.05
    ba = torch.from_numpy((rng.standard_normal((nframes, ncoeff)) + 1j * rng.standard_normal((nframes, ncoeff)))
                          .astype(np.complex64)).to(DEV)
    w = torch.from_numpy(rng.uniform(0.5, 1.5, coord.shape[:-1]).astype(np.float32))
    x = testing.complex_normal((coils, ncoeff) + (n,) * ndim, seed=1).to(DEV)
    y = [tilenufft.fft.apply_nufft(x, tilenufft.fft.plan_nufft(coord, n, 4, 1.5, device=DEV, interp_mode=m), ba, weight=w)
         for m in (1, 2)]
    assert float((y[0] - y[1]).abs().square().sum().sqrt() / y[0].abs().square().sum().sqrt()) < 1e-6
