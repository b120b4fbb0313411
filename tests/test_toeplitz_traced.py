"""Which calls of the Toeplitz operator native code can serve: those whose
tensors have memory of their own. Compilation, fake, proxy and functional
tensors, functorch transforms and subclasses with a dispatch of their own take
torch's calls; a mode that only watches changes nothing."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.testing._internal.two_tensor import TwoTensor
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.flop_counter import FlopCounterMode

from tilenufft import _core, testing
from tilenufft.fft.toeplitz import GramMatrix, apply_nufft_selfadj


class Watch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_traced():
    x = torch.ones(3)
    seen = []

    def f(y):
        seen.append(_core.traced(x, y))
        return (y * y).sum()

    def said(run):
        seen.clear()
        run()
        return set(seen)

    assert said(lambda: f(x)) == {False}
    assert said(lambda: f(torch.nn.Parameter(x))) == {False}
    assert said(lambda: torch.jit.trace(f, (x,), check_trace=False)) == {False}
    with FlopCounterMode(display=False), Watch():
        assert said(lambda: f(x)) == {False}
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert said(lambda: f(x)) == {True}
        fake = mode.from_tensor(x)
    assert said(lambda: f(fake)) == {True}
    assert said(lambda: make_fx(f)(x)) == {True}
    assert said(lambda: f(TwoTensor(x, x))) == {True}
    assert said(lambda: f(torch._to_functional_tensor(x))) == {True}
    for transform in (torch.func.grad(f), torch.func.functionalize(f), lambda y: torch.func.vmap(f)(y[None])):
        assert said(lambda: transform(x)) == {True}
    flag = torch.compile(lambda y: y + 1 if _core.traced(y) else y - 1, backend="eager", fullgraph=True)
    assert torch.equal(flag(x), x + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["compile", "fullgraph", "func.grad", "make_fx", "fake", "watch", "jit"])
def test_operator_under_tracers(how):
    """Values and gradients under each, against the plain call: torch's steps and
    the fused stages are each within the bound of two forward and two inverse
    line transforms (2 (2 11 + 6) 2^-24 per axis) of the 64-bit result."""
    print(f"toeplitz operator under {how}", flush=True)
    dev = "cuda:0"
    kern = GramMatrix(testing.complex_normal((64, 48), seed=1).to(dev), (64, 48), 2, dev, False)
    x = torch.view_as_real(testing.complex_normal((3, 32, 24), seed=2)).to(dev)
    tol = 2 * 2 * 2 * (2 * 11 + 6) * 2.0**-24

    def f(y):
        return torch.view_as_real(apply_nufft_selfadj(torch.view_as_complex(y), kern))

    ref = f(x)
    if how in ("compile", "fullgraph"):
        out = torch.compile(f, backend="eager", fullgraph=how == "fullgraph")(x)
    elif how == "func.grad":
        out = torch.func.grad(lambda y: 0.5 * (f(y) * y).sum())(x)
        leaf = x.clone().requires_grad_()
        (0.5 * (f(leaf) * leaf).sum()).backward()
        ref = leaf.grad
    elif how == "make_fx":
        out = make_fx(f)(x)(x)
    elif how == "fake":
        with FakeTensorMode(allow_non_fake_inputs=True) as mode:
            assert f(mode.from_tensor(x)).shape == ref.shape
        return
    elif how == "watch":
        with Watch():
            assert torch.equal(f(x), ref)  # the same stages
        return
    else:
        traced = torch.jit.trace(f, (torch.zeros_like(x),), check_trace=False)
        assert torch.equal(traced(x), ref)
        return
    assert float((out - ref).norm() / ref.norm()) < tol
