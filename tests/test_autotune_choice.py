"""The autotuner's choice (CPU only, with a clock in place of the device): the
gridding variant whose whole adjoint is fastest, also where another one's
gridding by itself is faster, and no choice cached for other kernels."""

import contextlib
import json
import types

import pytest
import torch

from tilenufft import autotune

GRIDDING = {0: 172.0, 3: 170.0, 2: 560.0, 1: 3600.0}
STAGES = {0: 352.0, 3: 390.0, 2: 352.0, 1: 352.0}


class Clocked:
    now = 0.0

    def __init__(self, plans, ncoils):
        self.mode, self.grid = plans[0].grid_mode, None

    def gridding(self, grid):
        Clocked.now += GRIDDING[self.mode]

    def adjoint(self):
        Clocked.now += GRIDDING[self.mode] + STAGES[self.mode]

    def interp(self, grid):
        Clocked.now += 100.0


def timed(fn, reps, device):
    start = Clocked.now
    fn()
    return Clocked.now - start


@pytest.fixture
def plans(monkeypatch, tmp_path):
    plan = types.SimpleNamespace(ndim=2, shape=(64, 64), os_shape=(128, 128), width=(4, 4), npts=1000, nframes=1,
                                 grid_mode=0)
    plan.interpolator = types.SimpleNamespace(device="cpu", grid_mode_effective=lambda: plan.grid_mode or 4)
    monkeypatch.setattr(autotune, "retune", lambda p, grid_mode=None, **kw: setattr(p, "grid_mode", grid_mode))
    monkeypatch.setattr(autotune, "BatchedNUFFT", Clocked)
    monkeypatch.setattr(autotune, "_time", timed)
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setenv("TILENUFFT_CACHE", str(tmp_path))
    return [plan]


def test_variant_of_the_fastest_adjoint(plans):
    best = autotune.tune_batch(plans, 4)
    assert best["grid_mode"] == 0 and plans[0].grid_mode == 0 and not best["cached"]
    assert best["grid_ms"] == GRIDDING[0]
    assert ("tile", (0, (32, 16)), GRIDDING[0] + STAGES[0]) in best["trials"]
    again = autotune.tune_batch(plans, 4)
    assert again["cached"] and again["grid_mode"] == 0


def test_choices_of_other_kernels_are_not_used(plans, tmp_path):
    autotune.tune_batch(plans, 4)
    path = tmp_path / "autotune.json"
    (key, value), = json.loads(path.read_text()).items()
    tag = f"|k{autotune._GENERATION}"
    assert key.count(tag) == 1
    for other in (key.replace(tag, ""), key.replace(tag, f"|k{autotune._GENERATION - 1}")):
        path.write_text(json.dumps({other: dict(value, grid_mode=3)}))
        best = autotune.tune_batch(plans, 4)
        assert not best["cached"] and best["grid_mode"] == 0
