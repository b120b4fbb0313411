"""One plan on several streams at once: hot tiles are split over workgroups,
whose partial sums each call keeps in a workspace of its own. Every result
equals the one of the calls in turn (same bits)."""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import _core, _lib, testing

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def hot(ndim, frames=1):
    rng = np.random.default_rng(3)
    return rng.normal(0, 1.5, (frames, 4, 100000, ndim)).clip(-16, 16).astype(np.float32)


@pytest.mark.parametrize("ndim, coils, lowrank, mode", [(2, 1, 0, 0), (2, 3, 0, 0), (3, 1, 0, 0), (2, 1, 4, 0),
                                                        (2, 1, 0, 3)])
def test_adjoints_of_one_plan_overlap(ndim, coils, lowrank, mode):
    print(f"streams {ndim}D coils={coils} lowrank={lowrank} grid_mode={mode}", flush=True)
    frames = 5 if lowrank else 1
    plan = tilenufft.fft.plan_nufft(hot(ndim, frames), 32, 4, 2.0, device=DEV, grid_mode=mode)
    basis = testing.complex_normal((lowrank, frames), seed=1).to(DEV) if lowrank else None
    lead = (coils, frames) if frames > 1 else (coils,)
    ys = [testing.complex_normal((*lead, 4, 100000), seed=10 + k).to(DEV) for k in range(6)]
    ref = [tilenufft.fft.apply_nufft_adj(y, plan, basis=basis) for y in ys]
    native = plan.interpolator if not lowrank else plan.lowrank_native
    assert native._workspaces[coils, lowrank] > 0
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = []
    for turn in range(12):
        for s, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                k = (turn + 2 * s) % len(ys)
                outs.append((k, tilenufft.fft.apply_nufft_adj(ys[k], plan, basis=basis)))
    torch.cuda.synchronize()
    for k, x in outs:
        assert torch.equal(torch.view_as_real(x), torch.view_as_real(ref[k]))


def test_workspace_need_and_own_workspace():
    """tn_grid and tn_grid_ws with and without a workspace give the same bits."""
    lib = _lib.load()
    plan = tilenufft.fft.plan_nufft(hot(2), 32, 4, 2.0, device=DEV)
    h, k = plan.interpolator.handle, testing.complex_normal((2, plan.npts), seed=5).to(DEV)
    print("workspace of the caller's", flush=True)
    with torch.cuda.device(DEV):
        need = lib.tn_plan_workspace(h, 2, 0)
        assert need > 0 and lib.tn_plan_workspace(h, 0, 0) == -1 and lib.tn_plan_workspace(h, 2**30, 2) == -4
        ws = torch.full((need,), float("nan"), device=DEV)
        grids = []
        for call in ("tn_grid", None, ws):
            g = torch.full((2, *plan.os_shape), float("nan"), dtype=torch.complex64, device=DEV)
            if call == "tn_grid":
                rc = lib.tn_grid(h, _core.ptr(k), _core.ptr(g), 2, None, _core.stream_ptr(DEV))
            else:
                rc = lib.tn_grid_ws(h, _core.ptr(k), _core.ptr(g), 2, None, _core.ptr(call), _core.stream_ptr(DEV))
            _lib.check(rc)
            grids.append(torch.view_as_real(g))
        torch.cuda.synchronize()
    assert torch.equal(grids[0], grids[1]) and torch.equal(grids[0], grids[2])


def test_tables_hold_partial_sums_only_for_calls_without_a_workspace():
    """The Python calls leave the launch tables without partial sums; the first
    call that brings no workspace, and tn_plan_prepare, allocate them once."""
    print("tables without partial sums", flush=True)
    lib = _lib.load()
    k = testing.complex_normal((3, 400000), seed=6).to(DEV)
    for prepare in (False, True):
        plan = tilenufft.fft.plan_nufft(hot(2), 32, 4, 2.0, device=DEV)
        native = plan.interpolator
        x = tilenufft.fft.apply_nufft_adj(k.reshape(3, 4, 100000), plan)
        tilenufft.fft.apply_nufft(x, plan)
        lean, need = native.device_bytes(), 4 * native._workspaces[3, 0]
        assert need > 0
        for _ in range(2):
            if prepare:
                native.prepare(3)
            else:
                g = torch.empty((3, *plan.os_shape), dtype=torch.complex64, device=DEV)
                with torch.cuda.device(DEV):
                    _lib.check(lib.tn_grid(native.handle, _core.ptr(k), _core.ptr(g), 3, None, _core.stream_ptr(DEV)))
                    torch.cuda.synchronize()
            assert native.device_bytes() == lean + need
