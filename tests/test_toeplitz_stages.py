"""The Toeplitz operator's FFT stages live as long as the operator: a captured
graph holds the device addresses of the stages that it was captured with, so
other shapes must not free them. On the CPU with stages that hold no device
memory in place of the native ones."""

import copy
import gc
import weakref

import pytest
import torch

from tilenufft import _core, testing
from tilenufft.fft.toeplitz import GramMatrix, apply_nufft_selfadj


class HostStages:
    def __init__(self, shape):
        self.shape = shape


def test_stages_of_every_shape_are_kept(monkeypatch):
    monkeypatch.setattr(_core, "fft_stages", lambda shape, grid, device: HostStages(shape) if shape[0] != 7 else None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    kern = GramMatrix(torch.ones(64, 64, dtype=torch.complex64), (64, 64), 2, "cpu", False)
    dev = torch.device("cpu")
    first = kern.stages((32, 32), dev)
    alive = weakref.ref(first)
    first = id(first)
    for n in range(3, 20):
        st = kern.stages((n, n), dev)
        assert (st is None) == (n == 7) and kern.stages((n, n), dev) is st
    gc.collect()
    assert alive() is not None and id(kern.stages((32, 32), dev)) == first
    assert "_stages" not in copy.deepcopy(kern).__dict__  # copies build their own
    kern.__dict__.clear()
    gc.collect()
    assert alive() is None


@pytest.mark.gpu
def test_replay_after_other_shapes():
    """Capture with one image shape, apply the same operator to others, replay:
    every replay equals the eager result of the same stages (same bits)."""
    print("toeplitz capture, other shapes, replay", flush=True)
    dev = "cuda:0"
    value = testing.complex_normal((96, 80), seed=1).to(dev)
    kern = GramMatrix(value, (96, 80), 2, dev, False)
    x = testing.complex_normal((2, 48, 40), seed=2).to(dev)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        apply_nufft_selfadj(x, kern)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = apply_nufft_selfadj(x, kern)
    for k, n in enumerate([(20, 31), (47, 40), (11, 80), (96, 33)]):
        apply_nufft_selfadj(testing.complex_normal((1, *n), seed=3).to(dev), kern)
        x.copy_(testing.complex_normal((2, 48, 40), seed=4 + k))
        graph.replay()
        assert torch.equal(y, apply_nufft_selfadj(x, kern))
