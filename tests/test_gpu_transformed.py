"""The NUFFT pair under functorch transforms, where the autograd functions are
bound by their signature, and outside of them, where a twin runs the same
forward and backward: the same gradients, bit for bit. Batching and
forward-mode differentiation, for which the functions have no rule, raise on
both routes."""

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwd

import tilenufft
from tilenufft import testing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("adjoint", [False, True])
def test_both_routes_agree(adjoint):
    rng = np.random.default_rng(3)
    coord = (rng.uniform(-0.5, 0.5, (1, 5, 61, 2)) * 24).astype(np.float32)
    plan = tilenufft.fft.plan_nufft(coord, 24, 4, 1.5, device=DEV)
    apply = tilenufft.fft.apply_nufft_adj if adjoint else tilenufft.fft.apply_nufft
    x = testing.complex_normal((2, 1, 5, 61) if adjoint else (2, 1, 24, 24), seed=1).to(DEV)

    def f(y):
        return apply(y, plan, device=DEV)

    print(f"transformed {apply.__name__}", flush=True)
    leaf = x.clone().requires_grad_()
    y = f(leaf)
    g = testing.complex_normal(tuple(y.shape), seed=2).to(DEV)
    y.backward(g)
    out, vjp = torch.func.vjp(f, x)
    assert torch.equal(torch.view_as_real(out), torch.view_as_real(y.detach()))
    assert torch.equal(torch.view_as_real(vjp(g)[0]), torch.view_as_real(leaf.grad))

    with pytest.raises(RuntimeError, match="vmap"):
        torch.func.vmap(f)(x[None])
    with pytest.raises(NotImplementedError, match="forward mode"):
        torch.func.jvp(f, (x,), (x,))
    with fwd.dual_level(), pytest.raises(NotImplementedError, match="forward mode"):
        f(fwd.make_dual(x, x))
