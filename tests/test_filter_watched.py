"""The row filter's kernel is used only for tensors that nothing follows (it is no torch operation): which tensors those
are (here), and that traces of ``filtering`` filter what they are given later (GPU)."""
import importlib

import numpy as np
import pytest
import torch

from tigre_amd.geometry import cone_geometry

F = importlib.import_module("tigre_amd.utilities.filtering")


def _seen(run):
    """What _unwatched says of the tensor that ``run`` hands to a function it follows."""
    said = []

    def f(x):
        said.append(F._unwatched(x))
        return x * 2.0

    run(f, torch.ones(3))
    assert said
    return said


def _dual(f, x):
    with torch.autograd.forward_ad.dual_level():
        f(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))


def _fx(f, x):
    from torch.fx.experimental.proxy_tensor import make_fx

    make_fx(f)(x)


def _fake(f, x):
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode() as mode:
        f(mode.from_tensor(x))


FOLLOWED = {
    "gradient": lambda f, x: f(x.requires_grad_()),
    "forward mode": _dual,
    "vmap": lambda f, x: torch.func.vmap(f)(x),
    "jvp": lambda f, x: torch.func.jvp(f, (x,), (x,)),
    "grad": lambda f, x: torch.func.grad(lambda y: f(y).sum())(x),
    "trace": lambda f, x: torch.jit.trace(f, (x,), check_trace=False),
    "make_fx": _fx,
    "fake": _fake,
    "parameter": lambda f, x: f(torch.nn.Parameter(x, requires_grad=False)),
    "negative view": lambda f, x: f(torch._neg_view(x)),
    "sparse": lambda f, x: f(x.to_sparse()),
}


@pytest.mark.parametrize("name", FOLLOWED)
def test_followed_tensors(name):
    assert not any(_seen(FOLLOWED[name]))


def test_plain_tensors():
    assert all(_seen(lambda f, x: f(x)))
    assert all(_seen(lambda f, x: f(x.expand(2, 3)[:, ::2])))

    def unrecorded(f, x):
        with torch.no_grad():
            f(x.requires_grad_())

    assert all(_seen(unrecorded))


@pytest.mark.parametrize("name", ["_functorch", "_len_torch_dispatch_stack"])
def test_missing_private_names(monkeypatch, name):
    monkeypatch.delattr(torch._C, name)
    assert not F._unwatched(torch.ones(3))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["jit", "fx"])
def test_traced_filter(cuda, kind):
    """A trace holds the operations, not the traced call's rows: the same numbers as a call, to the 3e-6 that the kernel
    and the padded transform may differ by."""
    geo = cone_geometry((4, 4, 4), (4.0, 4.0, 4.0), (3, 100), (1.0, 0.7), 300.0, 450.0)
    angles = np.linspace(0, 6, 5)
    geo.check_geo(angles)
    g = torch.Generator(device="cuda").manual_seed(1)
    first, second = (torch.randn((5, 3, 100), generator=g, device=cuda) for _ in range(2))

    def f(x):
        return F.filtering(x, geo, angles)

    if kind == "jit":
        traced = torch.jit.trace(f, (first,), check_trace=False)
    else:
        from torch.fx.experimental.proxy_tensor import make_fx

        traced = make_fx(f)(first)
    got, want = traced(second), f(second)
    assert float((got - want).norm() / want.norm()) <= 3e-6
