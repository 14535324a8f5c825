"""Row kernels at the widths where the number of chunks that a thread holds
changes, against float64.

Bounds: bf16 results are rounded (2^-9 of them; the sum of squares of at most
16384 floats and the reciprocal root add less than 2^-12); e4m3 results are the
scale times a value rounded to 3 bits of mantissa (2^-4 of it, and half of the
smallest step, 2^-10 of the scale)."""

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _rows(rows, width, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(rows, width, generator=g).bfloat16()


def _close(out, ref, quantised=False):
    if quantised:
        scale = out.scale.double().cpu()[:, None]
        out, bound = out.data.double().cpu() * scale, \
            ref.abs() * 2.0 ** -4 + scale * 2.0 ** -10
        assert torch.allclose(scale[:, 0], ref.abs().amax(-1) / 448,
                              rtol=2.0 ** -10)
    else:
        out, bound = out.double().cpu(), ref.abs() * 2.0 ** -8
    assert ((out - ref).abs() <= bound).all()


@pytest.mark.parametrize("hidden", [8, 4096, 4104, 8192, 8200, 16384])
def test_norms(hidden):
    x, r, w = (_rows(n, hidden, n) for n in (3, 3, 1))
    w = w[0]

    def ref(y):
        y = y.double()
        return y / (y.square().mean(-1, keepdim=True) + 1e-5).sqrt() \
            * w.double()

    gx, gr, gw = x.to(DEV), r.to(DEV), w.to(DEV)
    _close(ops.rmsnorm(gx, gw, 1e-5), ref(x))
    _close(ops.quant_fp8(gx), x.double(), True)
    both = x.double() + r.double()
    q, res = ops.fused_add_rmsnorm_q(gx, gr.clone(), gw, 1e-5)
    _close(q, ref(both), True)
    _close(res, both)
    y, res = ops.fused_add_rmsnorm(gx.clone(), gr.clone(), gw, 1e-5)
    _close(y, ref(both))
    _close(res, both)


@pytest.mark.parametrize("inter", [8, 8192, 8200, 16384, 16392, 32768])
def test_activation_in_e4m3(inter):
    x = _rows(3, 2 * inter, 7)
    g, u = x.double().split(inter, -1)
    _close(ops.silu_mul_q(x.to(DEV)), g * g.sigmoid() * u, True)


@pytest.mark.parametrize("parts", [2, 3, 5, 8])
@pytest.mark.parametrize("hidden", [8, 2048, 2056, 4096, 4104, 8192])
def test_norm_of_parts(hidden, parts):
    """The same bits as the sum, in order, and then the norm."""
    g = torch.Generator().manual_seed(hidden)
    part = torch.randn(parts, 5, hidden, generator=g).to(DEV)
    r, w = _rows(5, hidden, 1).to(DEV), _rows(1, hidden, 2)[0].to(DEV)
    total = part[0].clone()
    for z in range(1, parts):
        total += part[z]
    y, res = ops.fused_add_rmsnorm(total.bfloat16(), r.clone(), w, 1e-5)
    out = ops.fused_add_rmsnorm(ops.Parts(part), r, w, 1e-5)
    assert torch.equal(out[0], y) and torch.equal(out[1], res)


@pytest.mark.parametrize("rows", [16, 32, 200])
def test_parts_of_a_product(rows):
    x, w = _rows(rows, 4096, 3).to(DEV), _rows(4096, 4096, 4).to(DEV)
    out = ops.linear_parts(x, w)
    assert isinstance(out, ops.Parts) == (rows > 16)
    if rows > 16:
        out = out.data
        for z in range(1, len(out)):
            out[0] += out[z]
        out = out[0].bfloat16()
    assert torch.equal(out, ops.linear(x, w))


@pytest.mark.parametrize("hidden", [128, 2048, 2176, 4096, 4224, 8192])
@pytest.mark.parametrize("top", [1, 4, 5])
def test_norm_of_choices(hidden, top):
    """The same bits as the sum of the choices, then the norm."""
    g = torch.Generator().manual_seed(hidden + top)
    rows = 6
    data = _rows(rows * top + 3, hidden, 1).to(DEV)
    place = torch.randperm(rows * top, generator=g).int().view(rows, top)
    place[0, 0] = place[3] = -1
    place = place.to(DEV)
    weight = torch.rand(rows, top, generator=g).to(DEV)
    r, w = _rows(rows, hidden, 2).to(DEV), _rows(1, hidden, 3)[0].to(DEV)
    c = ops.Choices(data, place, weight)
    ref = ops.fused_add_rmsnorm(ops._moe_sum(c), r.clone(), w, 1e-5)
    out = ops.fused_add_rmsnorm(c, r.clone(), w, 1e-5)
    assert all(torch.equal(a, b) for a, b in zip(out, ref))
