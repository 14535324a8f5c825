"""Products that gradients, tangents, transforms, traces and modes see are
torch's, also where a kernel is as good for the sizes."""

import pytest
import torch
import torch.utils.flop_counter

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops


def _operands(dev):
    g = torch.Generator().manual_seed(2)
    return (torch.randn(4, 1024, generator=g).bfloat16().to(dev),
            torch.randn(2048, 1024, generator=g).bfloat16().to(dev))


class _Marked(torch.Tensor):
    pass


def test_what_a_kernel_may_replace():
    x, w = _operands("cpu")
    p = torch.nn.Parameter(w, requires_grad=False)
    assert ops.unrecorded(x, w) and ops.unrecorded(x, p)
    assert not ops.unrecorded(x.as_subclass(_Marked), w)
    grad = w.clone().requires_grad_()
    assert not ops.unrecorded(x, grad)
    with torch.no_grad():
        assert ops.unrecorded(x, grad)
    with torch.autograd.forward_ad.dual_level():
        assert not ops.unrecorded(x, w)
    with torch.autocast("cuda", dtype=torch.float16, enabled=True):
        on = torch.is_autocast_enabled("cuda")    # not without a GPU
        assert ops.unrecorded(x, w) != on
    with torch.utils.flop_counter.FlopCounterMode(display=False):
        assert not ops.unrecorded(x, w)
    seen = []
    f = lambda t: (seen.append(ops.unrecorded(t, w)), t * 2)[1]
    torch.func.vmap(f)(x)
    torch.jit.trace(f, x, check_trace=False)
    assert seen == [False] * len(seen) and len(seen) >= 2


@pytest.mark.gpu
def test_gradients_and_transforms_of_products():
    x, w = _operands("cuda:0")
    assert ops._plain_bf16(x, w) and ops._route(4, 2048, 1024, False) == "rows"
    ref = x.clone().requires_grad_()
    (ref @ w.t()).float().square().sum().backward()
    got = x.clone().requires_grad_()
    ops.linear(got, w).float().square().sum().backward()
    assert torch.equal(got.grad, ref.grad)
    out = torch.func.vmap(lambda t: ops.linear(t, w))(x[None].expand(3, 4, -1))
    assert out.shape == (3, 4, 2048)
    primal, tangent = torch.func.jvp(lambda t: ops.linear(t, w), (x,), (x,))
    assert torch.equal(primal, tangent)
    traced = torch.jit.trace(lambda t: ops.linear(t, w), x, check_trace=False)
    assert torch.equal(traced(2 * x), (2 * x) @ w.t())
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
