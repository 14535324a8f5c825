"""Products that gradients, tangents, transforms, traces and modes see are
torch's, also where a kernel is as good for the sizes."""

import warnings

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


class _Linear8(torch.nn.Module):
    def __init__(self, w, scale):
        super().__init__()
        self.w, self.scale = (torch.nn.Parameter(t, requires_grad=False)
                              for t in (w, scale))

    def forward(self, x, x_scale):
        return ops.linear_q(ops.QTensor(x, x_scale), self.w, self.scale)


def _operands8(rows, dev="cpu"):
    make = lambda *sizes: torch.empty(*sizes, dtype=torch.float8_e4m3fn,
                                      device=dev)
    return (make(rows, 1024), torch.ones(rows, device=dev), make(2048, 1024),
            torch.ones(2048, device=dev))


@pytest.mark.parametrize("dev", ["cpu", "cuda"])
def test_rows_that_are_a_symbol_stay_one(dev):
    """A product in 8 bits asks nothing about a number of rows without a value."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.symbolic_shapes import ShapeEnv
    with FakeTensorMode(shape_env=ShapeEnv()) as mode:   # no GPU, no memory
        rows = mode.shape_env.create_unbacked_symint()
        torch._check(rows >= 2)
        x, s, w, ws = _operands8(rows, dev)
        for parts in (False, True):
            y = ops.linear_q(ops.QTensor(x, s), w, ws, parts)
            assert y.shape[0] is rows or y.shape[0].node.expr == rows.node.expr


@pytest.mark.parametrize("rows", [8, 48, 200])
@pytest.mark.parametrize("strict", [False, True])
def test_export_of_any_number_of_rows(rows, strict):
    x, s, w, ws = _operands8(rows)
    n = torch.export.Dim("n", min=2, max=4096)
    out = torch.export.export(_Linear8(w, ws), (x, s), strict=strict,
                              dynamic_shapes=({0: n}, {0: n}))
    sizes = [v.meta["val"].shape[0] for v in out.graph.nodes
             if v.op == "call_function" and "_scaled_mm" in str(v.target)]
    assert len(sizes) == 1 and not isinstance(sizes[0], int)


def test_script_trace_of_rows_keeps_no_number(monkeypatch):
    monkeypatch.setattr(        # torch's has no scales of rows on the CPU
        torch, "_scaled_mm", lambda x, w, scale_a, scale_b, out_dtype:
        (x.float() * scale_a @ (w.float() * scale_b)).to(out_dtype))
    g = torch.Generator().manual_seed(3)
    draw = lambda *n: torch.randn(*n, generator=g)
    w, ws = draw(64, 32).to(torch.float8_e4m3fn), draw(64)
    x = draw(40, 32).to(torch.float8_e4m3fn)
    with warnings.catch_warnings():
        warnings.simplefilter("error", torch.jit.TracerWarning)
        traced = torch.jit.trace(_Linear8(w, ws), (x[:8], draw(8)),
                                 check_trace=False)
    s = draw(40)
    want = (x.float() * s[:, None] @ (w.float() * ws[:, None]).t()).bfloat16()
    assert torch.equal(traced(x, s), want)
