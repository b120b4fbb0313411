"""Batches of plans with different gridding variants and tap-record sizes:
which plans may share one, and results equal to the plans' own launches."""

import ctypes

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import _core, _lib, testing
from tilenufft.batch import BatchedNUFFT

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def coords(samples, n, seed, ndim=2):
    return np.random.default_rng(seed).uniform(-n / 2, n / 2, (1, samples, ndim)).astype(np.float32)


def test_one_batch_of_several_variants():
    """Tiles of both tap-record sizes (4 and 6 taps), the matrix as the
    automatic choice (7 taps) and as the one asked for, bit for bit."""
    lib = _lib.load()
    specs = [(4, 0, 3, 500), (6, 0, 9, 300), (7, 0, 2, 200), (4, 3, 1, 400), (5, 0, 17, 100)]
    plans = [tilenufft.fft.plan_nufft(coords(m, 30, s), 30, w, 1.5, device=DEV, grid_mode=mode)
             for s, (w, mode, _, m) in enumerate(specs)]
    assert [p.interpolator.grid_mode_effective() for p in plans] == [4, 4, 3, 3, 4]
    nb = [c for _, _, c, _ in specs]
    cells = int(np.prod(plans[0].os_shape))
    go = np.cumsum([0] + [c * cells for c in nb])
    so = np.cumsum([0] + [c * p.npts for c, p in zip(nb, plans)])
    arr = [(ctypes.c_int64 * len(nb))(*[int(v) for v in x]) for x in (nb, go[:-1], so[:-1])]
    handles = (ctypes.c_void_p * len(nb))(*[p.interpolator.handle.value for p in plans])
    out = ctypes.c_void_p()
    print("batch of several gridding variants", flush=True)
    with torch.cuda.device(DEV):
        _lib.check(lib.tn_batch_create(handles, *arr, None, len(nb), ctypes.byref(out)), "tn_batch_create")
        k = testing.complex_normal((int(so[-1]),), seed=1).to(DEV)
        grid = torch.full((int(go[-1]),), float("nan"), dtype=torch.complex64, device=DEV)
        _lib.check(lib.tn_batch_grid(out, _core.ptr(k), _core.ptr(grid), None, _core.stream_ptr(DEV)), "tn_batch_grid")
        back = torch.full_like(k, float("nan"))
        _lib.check(lib.tn_batch_interp(out, _core.ptr(grid), _core.ptr(back), None, _core.stream_ptr(DEV)),
                   "tn_batch_interp")
        torch.cuda.synchronize()
    for q, p in enumerate(plans):
        g = torch.empty((nb[q], *p.os_shape), dtype=torch.complex64, device=DEV)
        p.interpolator.gridding(k[so[q]:so[q + 1]].contiguous(), g, nb[q])
        assert torch.equal(torch.view_as_real(g.reshape(-1)), torch.view_as_real(grid[go[q]:go[q + 1]]))
        y = torch.empty((nb[q], p.npts), dtype=torch.complex64, device=DEV)
        p.interpolator.interp(g, y, nb[q])
        assert torch.equal(torch.view_as_real(y.reshape(-1)), torch.view_as_real(back[so[q]:so[q + 1]]))
    _lib.check(lib.tn_batch_destroy(out), "tn_batch_destroy")


def test_which_plans_share_a_batch():
    print("batch: automatic plans beyond the matrix, register runs asked for", flush=True)
    c = coords(15_000_000, 64, 7)  # x 36 taps x 8 bytes: more than the matrix may take
    big = tilenufft.fft.plan_nufft(c, 64, 6, 2.0, device=DEV)
    small, runs, spread, matrix = (tilenufft.fft.plan_nufft(coords(200, 64, 8), 64, 6, 2.0, device=DEV, grid_mode=m)
                                   for m in (0, 2, 1, 3))
    assert big.interpolator.grid_mode_effective() == 4
    for plans in ((big, runs), (runs, big), (big, small), (small, matrix), (matrix, small)):
        b = BatchedNUFFT(list(plans), 1)
        b.kspace.copy_(testing.complex_normal(b.kspace.shape, seed=2))
        b.gridding(b.grid)
        for q, p in enumerate(plans):
            g = torch.empty((1, *p.os_shape), dtype=torch.complex64, device=DEV)
            p.interpolator.gridding(b.kspace_view(q).reshape(1, -1).contiguous(), g, 1)
            assert torch.equal(torch.view_as_real(g[0]), torch.view_as_real(b.grid[q]))
    for plans in ((small, runs), (big, matrix), (runs, spread), (matrix, runs), (small, spread)):
        with pytest.raises(RuntimeError, match="share the gridding variant"):
            BatchedNUFFT(list(plans), 1)
