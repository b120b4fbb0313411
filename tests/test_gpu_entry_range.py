"""Tile entries beyond what 32-bit offsets hold: the tile gridding gives way to
the register runs, whose larger tiles make fewer entries, and those refuse what
is too many for them too. Plans only, nothing is transformed: every sample sits
at one point, whose footprint meets as many tiles as a footprint can (8)."""

import ctypes

import pytest
import torch

from tilenufft import _core, _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def plan(npts, at, mode, g=64):
    """(status, plan, coordinates) of a 3D plan of npts samples at (at, at, at)."""
    print(f"entry range: {npts} samples at {at}, grid_mode {mode}", flush=True)
    p = _lib.PlanParams()
    p.ndim, p.nframes, p.npts, p.grid_mode, p.inv_scale = 3, 1, npts, mode, 1.0
    p.shape[:], p.grid[:], p.width[:], p.beta[:] = [g // 2] * 3, [g] * 3, [4] * 3, [8.0] * 3
    coord = torch.full((npts, 3), float(at), device=DEV)
    handle = ctypes.c_void_p()
    with torch.cuda.device(DEV):
        rc = _lib.load().tn_plan_create(ctypes.byref(p), _core.ptr(coord), _core.stream_ptr(DEV), ctypes.byref(handle))
        torch.cuda.synchronize()
    return rc, handle


@pytest.mark.parametrize("mode", [0, 4])
def test_entries_beyond_32_bits(mode):
    lib = _lib.load()
    many = 2**28  # x 8 = 2^31 entries
    rc, handle = plan(many, 16, mode)  # origin 14: 8 tiles of 4^3 cells, and 8 of 16^3
    assert rc == -4 and "too many tile entries (2147483648)" in lib.tn_last_error().decode() and not handle.value
    rc, handle = plan(many, 4, mode)  # origin 2: 8 tiles of 4^3, one of 16^3
    assert rc == 0 and lib.tn_plan_grid_mode(handle) == 2 and lib.tn_plan_entries(handle) == many
    lib.tn_plan_destroy(handle)
    rc, handle = plan(1000, 16, mode)
    assert rc == 0 and lib.tn_plan_grid_mode(handle) == 4 and lib.tn_plan_entries(handle) == 8000
    lib.tn_plan_destroy(handle)
