"""Tile gridding of 48 MiB or more of samples, which reads a coil-minor copy of
them: each call keeps the copy in its own workspace, so that adjoints of one
plan may overlap on several streams, and a call without room for it reads the
samples in place. Same bits throughout."""

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import _core, _lib, testing

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
COILS, NPTS = 9, 700_001  # 48.07 MiB; one coil more than a block, ragged ends


def plan_of(ndim):
    rng = np.random.default_rng(ndim)
    coord = rng.uniform(-16, 16, (1, NPTS, ndim)).astype(np.float32)
    return tilenufft.fft.plan_nufft(coord, 32, 4, 2.0, device=DEV)


@pytest.mark.parametrize("ndim", [2, 3])
def test_adjoints_over_the_copy_overlap(ndim):
    print(f"streams over the copy {ndim}D", flush=True)
    plan = plan_of(ndim)
    ys = [testing.complex_normal((COILS, 1, NPTS), seed=10 + k).to(DEV) for k in range(3)]
    ref = [tilenufft.fft.apply_nufft_adj(y, plan) for y in ys]
    assert plan.interpolator.grid_mode_effective() == 4
    assert plan.interpolator._workspaces[COILS, 0] >= 2 * COILS * NPTS
    torch.cuda.synchronize()
    streams, outs = [torch.cuda.Stream() for _ in range(3)], []
    for turn in range(6):
        for s, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                k = (turn + s) % len(ys)
                outs.append((k, tilenufft.fft.apply_nufft_adj(ys[k], plan)))
    torch.cuda.synchronize()
    for k, x in outs:
        assert torch.equal(torch.view_as_real(x), torch.view_as_real(ref[k]))


@pytest.mark.parametrize("weighted", [False, True])
def test_with_and_without_room_for_the_copy(weighted):
    print(f"room for the copy weighted={weighted}", flush=True)
    lib, plan = _lib.load(), plan_of(2)
    native = plan.interpolator
    k = testing.complex_normal((COILS, NPTS), seed=5).to(DEV)
    w = torch.rand((1, NPTS), generator=torch.Generator().manual_seed(1)).to(DEV) if weighted else None
    out = []
    with torch.cuda.device(DEV):
        need = lib.tn_plan_workspace(native.handle, COILS, 0)
        lean = native.device_bytes()
        for call in ("workspace", "static", "own"):
            g = torch.full((COILS, *plan.os_shape), float("nan"), dtype=torch.complex64, device=DEV)
            args = (native.handle, _core.ptr(k), _core.ptr(g), COILS, _core.ptr(w))
            if call == "workspace":
                ws = torch.full((need,), float("nan"), device=DEV)
                _lib.check(lib.tn_grid_ws(*args, _core.ptr(ws), _core.stream_ptr(DEV)))
            else:
                _lib.check(getattr(lib, "tn_grid_static" if call == "static" else "tn_grid")(*args, _core.stream_ptr(DEV)))
            torch.cuda.synchronize()
            assert (native.device_bytes() > lean) == (call == "own")
            out.append(torch.view_as_real(g))
    assert native.device_bytes() - lean <= 4 * need
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
