"""Threads that meet at launch tables without buffers of their own: the first
calls that need them allocate them once, and every result has the bits of a
call by itself."""

import threading

import numpy as np
import pytest
import torch

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
THREADS = 6


def test_threads_allocate_once():
    rng = np.random.default_rng(3)
    coord = rng.normal(0, 1.5, (1, 4, 100000, 2)).clip(-16, 16).astype(np.float32)
    k = testing.complex_normal((2, 4, 100000), seed=6).to(DEV)
    for trial in range(5):
        print(f"threads, trial {trial}", flush=True)
        plan = tilenufft.fft.plan_nufft(coord, 32, 4, 2.0, device=DEV)
        native = plan.interpolator
        x = tilenufft.fft.apply_nufft_adj(k, plan)
        g = testing.complex_normal((2, *plan.os_shape), seed=trial).to(DEV)
        ref = torch.view_as_real(tilenufft.fft.apply_nufft(x, plan))
        lean, need = native.device_bytes(), 4 * native._workspaces[2, 0]
        assert need > 0
        outs = [torch.empty((2, plan.npts), dtype=torch.complex64, device=DEV) for _ in range(THREADS)]
        again = [None] * THREADS
        torch.cuda.synchronize()
        gate = threading.Barrier(THREADS)

        def work(q):
            with torch.cuda.device(DEV):
                gate.wait()
                native.interp(g, outs[q], 2)
                again[q] = torch.view_as_real(tilenufft.fft.apply_nufft(x, plan))

        threads = [threading.Thread(target=work, args=(q,)) for q in range(THREADS)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert native.device_bytes() == lean + need
        for q in range(THREADS):
            assert torch.equal(torch.view_as_real(outs[q]), torch.view_as_real(outs[0])) and torch.equal(again[q], ref)
