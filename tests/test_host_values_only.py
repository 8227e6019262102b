"""When a kernel may read a tensor's memory in place of tensor ops."""

import torch
import torch.autograd.forward_ad as fwAD
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

from mk._common import values_only


def test_values_only():
    a, seen = torch.ones(3), []

    def f(t):
        seen.append(values_only(t))
        return t * 2

    f(a)
    f(torch.nn.Parameter(a, requires_grad=False))
    g = a.clone().requires_grad_(True)
    with torch.no_grad():
        f(g)
    assert seen == [True, True, True]
    del seen[:]
    f(g)
    with fwAD.dual_level():
        f(fwAD.make_dual(a, a))
    torch.func.jvp(f, (a,), (a,))
    torch.func.vmap(f)(a)
    torch.func.vmap(lambda t: f(a) * t)(a)  # not a tensor of the transform's, but inside it
    torch.func.grad(lambda t: f(t).sum())(a)
    torch.jit.trace(f, (a,), check_trace=False)
    make_fx(f)(a)
    with FakeTensorMode() as mode:
        f(mode.from_tensor(a))
    assert seen and not any(seen)
