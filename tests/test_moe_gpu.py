"""Router kernel and grouped experts at both sides of the rules that choose
tiles of 16, 64, 128 and 256 rows, against float64.

Bounds: the router's products are exact in float and summed in float (2^-22 of
the sum of magnitudes); experts round their inner activation and their output
to bf16 (2^-9 each)."""

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("tokens,experts,top,width", [
    (1, 8, 2, 4096), (3, 64, 6, 2048), (65, 5, 5, 264), (2, 1, 1, 8),
    (7, 32, 4, 8200)])
def test_router(tokens, experts, top, width, fp8):
    g = torch.Generator().manual_seed(width)
    x = torch.randn(tokens, width, generator=g).bfloat16().to(DEV)
    router = torch.randn(experts, width, generator=g).bfloat16().to(DEV)
    arg = x
    if fp8:
        arg = ops.quant_fp8(x)
        x = (arg.data.float() * arg.scale[:, None]).bfloat16()
    weight, ids = ops.moe_router(arg, router, top)
    z = x.double() @ router.double().t()
    slack = 2.0 ** -22 * (x.double().abs() @ router.double().abs().t()).max()
    best = z.topk(top, -1)
    got = z.gather(1, ids.long())
    assert (got - best.values).abs().max() <= 2 * slack
    assert all(len(set(r)) == top for r in ids.tolist())
    ref = got.softmax(-1)
    assert (weight.double() - ref).abs().max() <= 4 * slack + 1e-6


@pytest.mark.parametrize("tokens", [1, 2, 12, 13, 64, 104, 105, 160, 161, 224, 225, 416,
                                    600])
@pytest.mark.parametrize("experts,top,width,inner", [
    (4, 2, 256, 128), (8, 1, 128, 384), (2, 2, 384, 32768)])
def test_experts_around_the_rule(tokens, experts, top, width, inner):
    g = torch.Generator().manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=g)
    x = rand(tokens, width).bfloat16().to(DEV)
    w13 = (rand(experts, 2 * inner, width) * width ** -0.5).bfloat16().to(DEV)
    w2 = (rand(experts, width, inner) * inner ** -0.5).bfloat16().to(DEV)
    # one expert may have no row, another most of them
    score = rand(tokens, experts)
    score[:, 0] += 1
    score[:, -1] -= 2
    ids = score.topk(top, -1).indices.int().to(DEV)
    weight = rand(tokens, top).abs().to(DEV)
    out = ops.moe_ffn(x, w13, w2, weight, ids).double()
    ref = torch.zeros_like(out)
    for e in range(experts):
        gate, up = (x.double() @ w13[e].double().t()).chunk(2, -1)
        y = torch.nn.functional.silu(gate) * up @ w2[e].double().t()
        ref += y * (weight * (ids == e)).sum(-1)[:, None].double()
    assert (out - ref).norm() <= 2.0 ** -7 * ref.norm()
    assert (out - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


def test_tiles_of_the_mean_of_choices():
    """Beyond 80 an expert, tiles of 256 rows, which are as high as their choices."""
    assert [ops._moe_tile(t, 2, 8, 16) for t in (11, 12, 192, 193, 320, 321, 448)] \
        == [16, 64, 64, 128, 128, 256, 256]
    assert ops._moe_tile(11, 2, 8, 64) == 64


@pytest.mark.parametrize("counts", [(256, 257, 0, 1), (1, 512, 200, 255),
                                    (96, 32, 64, 0), (97, 32, 64, 0)])
@pytest.mark.parametrize("width,inner", [(256, 32768), (384, 640)])
def test_tiles_of_one_and_of_several(counts, width, inner):
    """Experts of one tile, of several and of none, beside each other."""
    g = torch.Generator().manual_seed(sum(counts))
    rand = lambda *s: torch.randn(*s, generator=g)
    experts, tokens = len(counts), sum(counts)
    assert ops._moe_tile(tokens, 1, experts, 16) == (
        64 if tokens == 192 else 128 if tokens == 193 else 256)
    x = rand(tokens, width).bfloat16().to(DEV)
    w13 = (rand(experts, 2 * inner, width) * width ** -0.5).bfloat16().to(DEV)
    w2 = (rand(experts, width, inner) * inner ** -0.5).bfloat16().to(DEV)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])
    ids = ids[torch.randperm(tokens, generator=g)].int()[:, None].to(DEV)
    weight = rand(tokens, 1).abs().to(DEV)
    out = ops.moe_ffn(x, w13, w2, weight, ids).double()
    ref = torch.zeros_like(out)
    for e in range(experts):
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        gate, up = (x[rows].double() @ w13[e].double().t()).chunk(2, -1)
        y = torch.nn.functional.silu(gate) * up @ w2[e].double().t()
        ref[rows] = y * weight[rows].double()
    assert (out - ref).norm() <= 2.0 ** -7 * ref.norm()
    assert (out - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


@pytest.mark.parametrize("tokens,experts,top,width,inner", [
    (1, 4, 2, 128, 128), (5, 1, 1, 128, 256), (17, 4, 1, 256, 128),
    (33, 7, 1, 384, 640), (64, 64, 5, 128, 128), (65, 13, 1, 128, 384)])
@pytest.mark.parametrize("kind", ["spread", "one", "gaps"])
def test_few_choices(tokens, experts, top, width, inner, kind, monkeypatch):
    """Choices that are named where they are, more than 16 or 64 of one expert,
    and places without a choice."""
    monkeypatch.setattr(ops, "MOE_ROWS", 5)     # more than the rule gives it
    assert ops._moe_tile(tokens, top, experts, 16) == 16
    g = torch.Generator().manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=g)
    x = rand(tokens, width).bfloat16().to(DEV)
    w13 = (rand(experts, 2 * inner, width) * width ** -0.5).bfloat16().to(DEV)
    w2 = (rand(experts, width, inner) * inner ** -0.5).bfloat16().to(DEV)
    ids = rand(tokens, experts).topk(top, -1).indices.int()
    if kind == "one":
        ids[:, 0] = experts - 1
    elif kind == "gaps":
        ids[::3] = -1
    ids = ids.to(DEV)
    weight = rand(tokens, top).abs().to(DEV)
    out = ops.moe_ffn(x, w13, w2, weight, ids).double()
    ref = torch.zeros_like(out)
    for e in range(experts):
        gate, up = (x.double() @ w13[e].double().t()).chunk(2, -1)
        y = torch.nn.functional.silu(gate) * up @ w2[e].double().t()
        ref += y * (weight * (ids == e)).sum(-1)[:, None].double()
    assert (out - ref).norm() <= 2.0 ** -7 * ref.norm()
    assert (out - ref).abs().max() <= 2.0 ** -5 * ref.abs().max()


@pytest.mark.parametrize("up", [True, False])
@pytest.mark.parametrize("columns", [128, 1024, 1152, 2048, 2176, 4096, 6144])
def test_few_choices_and_where_their_columns_begin(up, columns):
    """Rows of multiples of 4 KB, whose workgroups begin at columns of their own, and
    others.  A sum is rounded to bf16, half a step being at most 2^-8 of it; a choice
    has the same bits alone."""
    E, N, T = 3, 256, 21
    g = torch.Generator().manual_seed(columns)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)
    x = rand(T, columns).bfloat16()
    w = (rand(E, (2 if up else 1) * N, columns) * columns ** -0.5).bfloat16()
    ids = (torch.arange(T) ** 2 % E).int().to(DEV)[:, None].contiguous()
    few = ops._native().experts_few
    out = torch.empty(T, N, dtype=torch.bfloat16, device=DEV)
    place = torch.empty_like(ids) if up else None
    few(up, out, place, x, w, ids, 1)
    for t in range(T):
        e = int(ids[t])
        want = w[e].double() @ x[t].double()
        slack = (w[e].double().abs() @ x[t].double().abs()) * 2.0 ** -22
        if up:
            # |silu'| <= 1.1, |silu(g)| <= |g|; the exponential's error is 2^-20
            (gate, v), (dg, dv) = want.chunk(2), slack.chunk(2)
            want = torch.nn.functional.silu(gate) * v
            slack = 1.1 * dg * v.abs() + gate.abs() * dv + 2.0 ** -20 * want.abs()
        assert ((out[t].double() - want).abs()
                <= 2.0 ** -8 * want.abs() + 1.01 * slack).all()
    one = torch.empty(1, N, dtype=torch.bfloat16, device=DEV)
    few(up, one, place[:1].clone() if up else None, x[20:], w, ids[20:].clone(), 1)
    assert torch.equal(one[0], out[20])


def test_choices_that_name_no_expert():
    """Without a sort: no place, and nothing of them in the sum; and no more
    experts than a load of their numbers has."""
    few = ops._native().experts_few
    x = torch.randn(6, 128, device=DEV).bfloat16()
    w = torch.randn(4, 256, 128, device=DEV).bfloat16()
    ids = torch.tensor([1, -1, 4, 3, 1 << 30, -(1 << 31)], dtype=torch.int32,
                       device=DEV)
    out = torch.full((6, 128), 7.0, device=DEV).bfloat16()
    place = torch.empty_like(ids)
    few(True, out, place, x, w, ids, 1)
    assert place.tolist() == [0, -1, -1, 3, -1, -1]
    assert (out[place < 0] == 7).all() and not (out[place >= 0] == 7).all(1).any()
    many = torch.randn(65, 256, 128, device=DEV).bfloat16()
    with pytest.raises(RuntimeError):
        few(True, out, place, x, many, ids, 1)


@pytest.mark.parametrize("tokens", [1, 26, 27, 56, 57, 300])
@pytest.mark.parametrize("experts,top,width,inner", [
    (4, 2, 256, 384), (3, 1, 1024, 256)])
def test_experts_with_8_bits(tokens, experts, top, width, inner):
    """Against float64 on the quantized operands.  The inner activation is
    rounded to e4m3: a step of at most 2^-3 of a value, 2^-4 / sqrt(3) of it on
    average, and of the sum of such."""
    from hyperspot.parallel.layers import quantize_weight_fp8
    g = torch.Generator().manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)
    xq = ops.quant_fp8(rand(tokens, width).bfloat16())
    w13, s13, w2, s2 = (torch.stack(t) for t in zip(*(
        quantize_weight_fp8(rand(2 * inner, width) * width ** -0.5)
        + quantize_weight_fp8(rand(width, inner) * inner ** -0.5)
        for _ in range(experts))))
    ids = rand(tokens, experts).topk(top, -1).indices.int()
    weight = rand(tokens, top).abs()
    out = ops.moe_ffn_fp8(xq, w13, s13, w2, s2, weight, ids).double()
    x = xq.data.double() * xq.scale.double()[:, None]
    ref = torch.zeros_like(out)
    for e in range(experts):
        gate, up = (x @ (w13[e].double() * s13[e].double()[:, None]).t()) \
            .chunk(2, -1)
        y = torch.nn.functional.silu(gate) * up \
            @ (w2[e].double() * s2[e].double()[:, None]).t()
        ref += y * (weight * (ids == e)).sum(-1)[:, None].double()
    assert (out - ref).norm() <= 2.0 ** -4.5 * ref.norm()


def test_refused_sizes():
    x = torch.zeros(3, 192, device=DEV).bfloat16()
    w13, w2 = (torch.zeros(2, *s, device=DEV).bfloat16()
               for s in ((256, 192), (192, 128)))
    ids = torch.zeros(3, 1, dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError):
        ops.moe_ffn(x, w13, w2, torch.ones(3, 1, device=DEV), ids)


@pytest.mark.parametrize("tokens", [1280, 1281])
@pytest.mark.parametrize("fp8", [False, True])
def test_many_tokens_over_many_experts(tokens, fp8, monkeypatch):
    """The kernel up to the rule's bound and torch's operations beyond it make
    the same choices, but for logits that are as close as float sums are."""
    from hyperspot.engine import ModelSpec
    from hyperspot.models.mixtral import MixtralMoE
    from hyperspot.parallel import layers
    monkeypatch.setattr(layers, "_QUANT_MODE", "fp8" if fp8 else None)
    monkeypatch.setattr(layers, "_INIT_DEVICE", DEV)
    spec = ModelSpec("m", 256, 1, 2, 1, 128, 128 if not fp8 else 256, 64,
                     num_experts=64, num_experts_per_tok=4)
    moe = MixtralMoE(spec, 0, torch.bfloat16).to(DEV)
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn(tokens, 256, generator=g).bfloat16().to(DEV)
    moe.router.data.copy_(torch.randn(64, 256, generator=g))
    seen = []
    kernel = ops._native().experts_router
    monkeypatch.setattr(ops._native(), "experts_router", lambda *a: (
        seen.append(1), kernel(*a))[1])
    xq = ops.quant_fp8(x) if fp8 else x
    out = moe(xq)
    assert len(seen) == (tokens == 1280)
    weight, ids = ops.moe_router(xq, moe.router, 4)
    ref = ops.moe_ffn_fp8(xq, moe.w13, moe.w13_scale, moe.w2, moe.w2_scale,
                          weight, ids) if fp8 \
        else ops.moe_ffn(x, moe.w13, moe.w2, weight, ids)
    same = (out.float() - ref.float()).abs() <= 2.0 ** -7 * ref.float().abs() \
        .max()
    assert same.all(-1).float().mean() >= 0.99


@pytest.mark.gpu
def test_rows_beyond_32_bits():
    """Tokens whose rows do not lie within 4 GB of the first one."""
    tokens, width, inner = (1 << 19) + 300, 4096, 128
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.empty(tokens, width, dtype=torch.bfloat16, device=DEV)
    x.normal_(generator=g)
    new = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16() * 0.02
    w13, w2 = new(2, 2 * inner, width), new(2, width, inner)
    ids = torch.randint(0, 2, (tokens, 1), generator=g, device=DEV,
                        dtype=torch.int32)
    ones = torch.ones(tokens, 1, device=DEV)
    out = ops.moe_choices(x, w13, w2, ones, ids)
    rows = torch.tensor([0, 1, 255, 1 << 18, (1 << 19) - 1, 1 << 19,
                         tokens - 1], device=DEV)
    got = out.data[out.place[rows, 0].long()]
    few = ops.moe_choices(x[rows], w13, w2, ones[rows], ids[rows])
    want = few.data[few.place[:, 0].long()].float()
    # both round the inner values and the results to bf16
    assert (got.float() - want).norm() <= 2.0 ** -7 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,experts,top,width,parts", [
    (1, 1, 1, 8, 0), (3, 16, 2, 2048, 0), (5, 17, 3, 2056, 2), (64, 33, 4, 4096, 8),
    (17, 64, 8, 8192, 3), (200, 8, 2, 4104, 0)])
def test_norm_and_router(tokens, experts, top, width, parts):
    """As the norm, then the router of what it gives."""
    g = torch.Generator().manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)
    x = ops.Parts(rand(parts, tokens, width)) if parts \
        else rand(tokens, width).bfloat16()
    res, norm = rand(tokens, width).bfloat16(), rand(width).bfloat16()
    router = (rand(experts, width) * width ** -0.5).bfloat16()
    got, got_res = ops.fused_add_rmsnorm_route(x, res.clone(), norm, 1e-5,
                                               router, top)
    h, want_res = ops.fused_add_rmsnorm(x if parts else x.clone(), res.clone(),
                                        norm, 1e-5)
    assert torch.equal(got_res, want_res)
    # the squares are added in another order: the last bit of a row's scale
    assert ((got.data.float() - h.float()).abs()
            <= h.float().abs() * 2.0 ** -7).all()
    # what the router makes of those rows is what it makes of them by itself
    weights, ids = ops.moe_router(got.data, router, top)
    assert torch.equal(got.ids, ids) and torch.equal(got.weights, weights)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,experts,top", [(4, 32, 4), (60, 4, 2), (200, 8, 2)])
def test_padding_chooses_no_expert(tokens, experts, top):
    """Without a sort and in tiles; the other rows are as without padding, and the
    padding's own get nothing from the experts."""
    g = torch.Generator().manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)
    W, I = 256, 128
    x, res, norm = (rand(tokens, W).bfloat16(), rand(tokens, W).bfloat16(),
                    rand(W).bfloat16())
    router = (rand(experts, W) * W ** -0.5).bfloat16()
    w13 = (rand(experts, 2 * I, W) * W ** -0.5).bfloat16()
    w2 = (rand(experts, W, I) * I ** -0.5).bfloat16()
    slots = torch.arange(tokens, device=DEV) - 1
    slots[tokens // 2:tokens * 3 // 4] = -1
    pad = slots < 0
    out = []
    for s in (None, slots):
        h, r = ops.fused_add_rmsnorm_route(x, res.clone(), norm, 1e-5, router,
                                           top, s)
        c = ops.moe_choices(h.data, w13, w2, h.weights, h.ids)
        out.append((h, *ops.fused_add_rmsnorm(c, r, norm, 1e-5), r))
    (h0, y0, r0, _), (h1, y1, r1, _) = out
    assert (h1.ids[pad] == -1).all() and (h1.weights[pad] == 0).all()
    assert torch.equal(h0.ids[~pad], h1.ids[~pad])
    assert torch.equal(h0.weights[~pad], h1.weights[~pad])
    assert torch.equal(h0.data, h1.data)
    assert torch.equal(y0[~pad], y1[~pad]) and torch.equal(r0[~pad], r1[~pad])
    # the first norm's sum, and nothing added
    assert torch.equal(r1[pad], (x.float() + res.float()).bfloat16()[pad])


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [5, 130])
@pytest.mark.parametrize("fp8", [False, True])
def test_padding_of_the_router(tokens, fp8):
    """By itself, and through the experts in 8 bits."""
    from hyperspot.parallel.layers import quantize_weight_fp8
    g = torch.Generator().manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)
    E, W, I, top = 4, 256, 256, 2
    x, router = rand(tokens, W).bfloat16(), rand(E, W).bfloat16()
    xq = ops.quant_fp8(x) if fp8 else x
    slots = torch.arange(tokens, device=DEV) % 4 - 1
    pad = slots < 0
    weight, ids = ops.moe_router(xq, router, top)
    got, got_ids = ops.moe_router(xq, router, top, slots)
    assert torch.equal(got[~pad], weight[~pad]) and (got[pad] == 0).all()
    assert torch.equal(got_ids[~pad], ids[~pad]) and (got_ids[pad] == -1).all()
    if not fp8:
        return
    w13, s13, w2, s2 = (torch.stack(t) for t in zip(*(
        quantize_weight_fp8(rand(2 * I, W) * W ** -0.5)
        + quantize_weight_fp8(rand(W, I) * I ** -0.5) for _ in range(E))))
    want = ops.moe_ffn_fp8(xq, w13, s13, w2, s2, weight, ids)
    out = ops.moe_ffn_fp8(xq, w13, s13, w2, s2, got, got_ids)
    assert torch.equal(out[~pad], want[~pad]) and (out[pad] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["", "moe"])
def test_watched_experts_get_tensors(path):
    from hyperspot.engine.config import ModelSpec
    from hyperspot.models.llama import DecoderLayer
    from hyperspot.models.mixtral import _MoEAdapter
    from hyperspot.parallel import layers
    layers.set_init_device(DEV)
    spec = ModelSpec("t", 256, 1, 2, 1, 128, 256, 32, num_experts=4,
                     num_experts_per_tok=2)
    layer = DecoderLayer(spec, 0, torch.bfloat16, _MoEAdapter).to(DEV)
    layers.set_init_device("cpu")
    x = torch.randn(6, 256, device=DEV).bfloat16()
    routed = []
    take = layer.mlp.moe._norm_router(x, x.clone(), layer.post_norm_w)
    assert take is not None and take[1] == 2
    layer.mlp.get_submodule(path).register_forward_hook(
        lambda m, a, y: routed.append(type(a[0])))
    assert layer.mlp._norm_router(x, x.clone(), layer.post_norm_w) is None \
        if path else layers.watched(layer.mlp)
    layer.mlp(x)
    assert routed == [torch.Tensor]


@pytest.mark.parametrize("width,inner", [(4096, 1024), (1024, 4096)])
def test_tiles_of_an_expert_together(width, inner):
    """Experts of 0 to 34 tiles of 256, beside each other up to 32."""
    counts = [8500, 1, 300, 0, 513, 256]
    g = torch.Generator(device=DEV).manual_seed(width)
    new = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    ids = torch.repeat_interleave(torch.arange(6, dtype=torch.int32),
                                  torch.tensor(counts))
    ids = ids[torch.randperm(len(ids))].to(DEV)
    x = new(len(ids), width)
    w13 = new(6, 2 * inner, width) * width ** -0.5
    w2 = new(6, width, inner) * inner ** -0.5
    out = ops.moe_ffn(x, w13, w2, torch.ones(len(ids), 1, device=DEV),
                      ids[:, None])
    for e in range(6):
        mine = ids == e
        gate, up = (x[mine].float() @ w13[e].float().t()).chunk(2, 1)
        want = (torch.nn.functional.silu(gate) * up) @ w2[e].float().t()
        # both round the inner values and the results to bf16
        assert (out[mine].float() - want).norm(dim=-1).le(
            2.0 ** -7 * want.norm(dim=-1)).all()


@pytest.mark.parametrize("kind", ["gated", "plain", "fp8"])
@pytest.mark.parametrize("outputs", [384, 2560])    # tiles of 128 and of 256
@pytest.mark.parametrize("chunks", [2, 3, 5])
def test_tiles_as_high_as_their_choices(kind, outputs, chunks):
    """Tiles of 1 to 8 blocks of 32 choices, at the edges of the blocks; experts of
    several tiles have even ones.  A sum is rounded to bf16: half a step is at most
    2^-8 of it."""
    counts = [1, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225,
              256, 257, 0, 300, 513]
    E, T, fp8 = len(counts), sum(counts), kind == "fp8"
    K = chunks * (128 if fp8 else 64)
    g = torch.Generator().manual_seed(chunks)
    rand = lambda *s: torch.randn(*s, generator=g).to(DEV)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(T, generator=g)].int().to(DEV)
    order, expert, place = ops._moe_sort(ids[:, None], E, 128, 128, 256)
    live = (order.view(-1, 256) >= 0).sum(1)
    for e, n in enumerate(counts):
        tiles = live[expert == e]
        assert int(tiles.sum()) == n and len(tiles) == -(-n // 256)
        assert n == 0 or int(tiles.max() - tiles.min()) < 32 * len(tiles)
    gated = kind == "gated"
    x, w = rand(T, K), rand(E, outputs, K) * K ** -0.5
    N = outputs // 2 if gated else outputs
    out = torch.empty(len(order), N, dtype=torch.bfloat16, device=DEV)
    sx = sw = None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        sx, sw = rand(T).abs(), rand(E, outputs).abs()
    else:
        x, w = x.bfloat16(), w.bfloat16()
    ops._native().experts_tiles(out, x, w, sx, sw, order, expert, gated, 1, 256)
    got = out[place[:, 0].long()].double()
    for e in range(E):
        mine = ids == e
        want = x[mine].double() @ w[e].double().t()
        # of a sum of magnitudes: float sums, and the 8-bit products of the card,
        # which keep fewer bits of a part of K
        slack = (x[mine].double().abs() @ w[e].double().abs().t()) \
            * 2.0 ** (-16 if fp8 else -22)
        if gated:
            gate, up = want.chunk(2, -1)
            want = torch.nn.functional.silu(gate) * up
            # |silu'| <= 1.1, |silu(g)| <= |g|; the exponential's error is 2^-20
            dg, du = slack.chunk(2, -1)
            slack = 1.1 * dg * up.abs() + gate.abs() * du \
                + 2.0 ** -20 * want.abs()
        if fp8:
            scale = sx[mine, None].double() * sw[e].double()
            want, slack = want * scale, slack * scale
        assert ((got[mine] - want).abs()
                <= 2.0 ** -8 * want.abs() + 1.01 * slack).all()


@pytest.mark.parametrize("kind", ["gated", "plain", "fp8"])
@pytest.mark.parametrize("outputs", [1152, 4096])   # tiles of 128 and of 256
@pytest.mark.parametrize("row_kb", [4, 6, 8])
def test_where_tiles_of_one_expert_begin(kind, outputs, row_kb):
    """Tiles of rows of 4 KB, and with gates of 8 KB, begin their weights at columns of
    their own, but not those of an expert that has two.  Bounds as above."""
    gated, fp8 = kind == "gated", kind == "fp8"
    counts = [130, 200, 256, 131, 257, 140, 180, 150, 222, 160]
    E, T = len(counts), sum(counts)
    K = row_kb * (1024 if fp8 else 512)
    rows = outputs * (2 if gated else 1)
    g = torch.Generator(DEV).manual_seed(row_kb)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).int().to(DEV)
    order, expert, place = ops._moe_sort(ids[:, None], E, 128, 128, 256)
    x, w = rand(T, K).bfloat16(), (rand(E, rows, K) * K ** -0.5).bfloat16()
    sx = sw = None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), (w * 64).to(torch.float8_e4m3fn)
        sx, sw = rand(T).abs(), rand(E, rows).abs()

    def product(w):
        out = torch.empty(len(order), outputs, dtype=torch.bfloat16, device=DEV)
        ops._native().experts_tiles(out, x, w, sx, sw, order, expert, gated, 1, 256)
        return out[place[:, 0].long()]

    got = product(w)
    for e in range(E):
        mine = ids == e
        a, b = x[mine].double(), w[e].double()
        want, slack = a @ b.t(), a.abs() @ b.abs().t() * 2.0 ** (-16 if fp8 else -22)
        if gated:
            (gate, up), (dg, du) = want.chunk(2, -1), slack.chunk(2, -1)
            want = torch.nn.functional.silu(gate) * up
            slack = 1.1 * dg * up.abs() + gate.abs() * du + 2.0 ** -20 * want.abs()
        if fp8:
            scale = sx[mine, None].double() * sw[e].double()
            want, slack = want * scale, slack * scale
        assert ((got[mine].double() - want).abs()
                <= 2.0 ** -8 * want.abs() + 1.01 * slack).all()
    if fp8:
        return
    # 256 outputs on, the same weights are another tile's; roundings hide most changes
    turned = w.view(E, 2 if gated else 1, outputs, K).roll(256, 2).reshape(w.shape)
    other = product(turned).roll(-256, 1)
    apart = (other != got).any(-1)
    alone = torch.tensor([n <= 256 for n in counts], device=DEV)[ids.long()]
    assert not apart[~alone].any()
    assert bool(apart[alone].any()) == (row_kb == 4 or row_kb == 8 and gated)
