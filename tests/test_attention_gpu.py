"""Prompt attention on the matrix cores: portions over the pages, and the
edges of tiles, against the PyTorch reference in float64.

Bounds: outputs are rounded to bf16 (2^-9 of the value) and are means of
values of about one; weights enter as three bf16 parts over the pages (the
bound is that of two, 2^-16) and as one (2^-9) beside q."""

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops
from hyperspot.models.llama import ForwardMeta

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
D = 128


def _reference(q, k, v, before, scale):
    """q [n, H, D] are the tokens after `before` of k, v [before + n, KV, D]."""
    n, group = q.shape[0], q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(group, 1) for t in (k, v))
    s = torch.einsum("qhd,khd->hqk", q.double().cpu(), k.cpu()) * scale
    seen = torch.arange(k.shape[0])[None] <= before + torch.arange(n)[:, None]
    s = s.masked_fill(~seen, float("-inf")).softmax(-1)
    return torch.einsum("hqk,khd->qhd", s, v.cpu())


def _check(out, ref, weight_step):
    err = (out.double().cpu() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + weight_step * 4
    assert (err <= bound).all(), float((err - bound).max())


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("group,kv", [(4, 2), (8, 1), (2, 3), (1, 2)])
@pytest.mark.parametrize("portions", [
    [(0, 16), (16, 17), (47, 63), (64, 1)],     # (before, rows)
    [(100, 130), (0, 64), (3, 15), (200, 32)],
    [(1, 257)], [(40, 79)], [(40, 80)],
])
def test_portions_over_pages(portions, group, kv, fp8):
    g = torch.Generator().manual_seed(3)
    heads, lens = group * kv, [n for _, n in portions]
    total = sum(lens)
    q = torch.randn(total, heads, D, generator=g).bfloat16().to(DEV)
    tables = [-(-(b + n) // 16) for b, n in portions]
    pages = sum(tables) + 3
    order = torch.randperm(pages, generator=g)
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    # what the last page holds after the last token is not a part of it
    kc, vc = (torch.randn(pages, kv, 16, D, generator=g).to(kind).to(DEV)
              for _ in range(2))
    bt = torch.zeros(len(portions), max(tables) + 1, dtype=torch.int32)
    at, starts, ctx, row_seq = 0, [0], [], []
    for i, (b, n) in enumerate(portions):
        bt[i, :tables[i]] = order[at:at + tables[i]]
        at += tables[i]
        starts.append(starts[-1] + n)
        ctx += range(b + 1, b + n + 1)
        row_seq += [i] * n
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    meta = ForwardMeta("prefill", None, None, seq_start=i32(starts),
                       max_seqlen=max(lens), row_seq=i32(row_seq),
                       ctx_lens=i32(ctx), block_tables=bt.to(DEV),
                       fresh_prefill=False)
    out = ops.attention(q, None, None, kc, vc, meta, D ** -0.5)
    for i, (b, n) in enumerate(portions):
        page = bt[i, :tables[i]].long().to(DEV)
        k, v = (c[page].float().transpose(1, 2).reshape(-1, kv, D)[:b + n]
                for c in (kc, vc))
        rows = slice(starts[i], starts[i] + n)
        _check(out[rows], _reference(q[rows], k, v, b, D ** -0.5), 2.0 ** -14)


@pytest.mark.parametrize("scale", [D ** -0.5, -0.2, 0.0])
@pytest.mark.parametrize("heads,kv", [(4, 1), (6, 2), (2, 1), (3, 3)])
@pytest.mark.parametrize("lens", [[1, 31, 32, 33], [64, 129, 0, 2], [200]])
def test_whole_prompts(lens, heads, kv, scale):
    g = torch.Generator().manual_seed(4)
    total = sum(lens)
    # columns of one buffer, as the projection leaves them
    qkv = torch.randn(total, (heads + 2 * kv) * D, generator=g) \
        .bfloat16().to(DEV)
    q, k, v = (t.view(total, -1, D) for t in
               qkv.split([heads * D, kv * D, kv * D], -1))
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    meta = ForwardMeta("prefill", None, None, max_seqlen=max(lens),
                       seq_start=torch.tensor(starts, dtype=torch.int32,
                                              device=DEV))
    out = ops.attention(q, k, v, k.new_empty(0, kv, 16, D), None, meta, scale)
    for a, b in zip(starts, starts[1:]):
        if a < b:
            _check(out[a:b], _reference(q[a:b], k[a:b], v[a:b], 0, scale),
                   2.0 ** -9)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("group,kv", [(1, 2), (2, 1), (3, 1), (4, 3), (8, 1)])
@pytest.mark.parametrize("split", [1, 2, 5, 64])
def test_decode_over_pages(split, group, kv, fp8):
    from hyperspot import _C
    g = torch.Generator().manual_seed(6)
    ctx = [1, 15, 16, 17, 32, 33, 127, 128, 129, 700]
    heads = group * kv
    q = torch.randn(len(ctx), heads, D, generator=g).bfloat16().to(DEV)
    tables = [-(-n // 16) for n in ctx]
    pages = sum(tables) + 3
    order = torch.randperm(pages, generator=g)
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    kc, vc = (torch.randn(pages, kv, 16, D, generator=g).to(kind).to(DEV)
              for _ in range(2))
    bt = torch.zeros(len(ctx), max(tables) + 1, dtype=torch.int32)
    at = 0
    for i, t in enumerate(tables):
        bt[i, :t] = order[at:at + t]
        at += t
    lens = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    out = torch.empty_like(q)
    ws = torch.empty(len(ctx) * heads * split * (D + 2), device=DEV) \
        if split > 1 else None
    _C.paged_attn(out, q, kc, vc, bt.to(DEV), lens, None, D ** -0.5, ws,
                  split)
    for i, n in enumerate(ctx):
        page = bt[i, :tables[i]].long().to(DEV)
        k, v = (c[page].float().transpose(1, 2).reshape(-1, kv, D)[:n]
                for c in (kc, vc))
        _check(out[i:i + 1], _reference(q[i:i + 1], k, v, n - 1, D ** -0.5),
               2.0 ** -14)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("group,kv", [(4, 2), (8, 1), (3, 2), (2, 3), (1, 4)])
@pytest.mark.parametrize("lens", [
    [1, 16, 17, 31, 32, 33], [127, 128, 129, 500, 2], [700],
    list(range(1, 131)),                        # one part
])
def test_rope_in_decode_attention(lens, group, kv, fp8):
    """Against the two launches: the same bytes in the pages; a row without a
    slot leaves them and attends over what they hold.  A turned value may fall
    on the other side of a rounding to bf16 (2^-8 of it, of outputs of about
    one)."""
    g = torch.Generator().manual_seed(5)
    n, heads = len(lens), group * kv
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    tables = [-(-x // 16) for x in lens]
    order = torch.randperm(sum(tables), generator=g).int()
    caches = [torch.randn(sum(tables), kv, 16, D, generator=g).to(kind).to(DEV)
              for _ in range(2)]
    bt = torch.zeros(n, max(tables), dtype=torch.int32)
    slots, at = [], 0
    for i, (x, t) in enumerate(zip(lens, tables)):
        bt[i, :t] = order[at:at + t]
        at += t
        slots.append(int(bt[i, t - 1]) * 16 + (x - 1) % 16 if i != 1 else -1)
    ang = torch.rand(1000, D // 2, generator=g) * 6.3
    cos_sin = torch.cat([ang.cos(), ang.sin()], -1).to(DEV)
    lens, slots = torch.tensor(lens), torch.tensor(slots).to(DEV)
    meta = ForwardMeta("decode", (lens - 1).to(DEV), slots,
                       block_tables=bt.to(DEV), seq_lens=lens.int().to(DEV))
    qkv = torch.randn(n, heads + 2 * kv, D, generator=g).bfloat16().to(DEV)
    outs, pages = [], []
    for fused in (True, False):
        kc, vc = (c.clone() for c in caches)
        q, k, v = qkv.clone().split([heads, kv, kv], 1)
        assert ops._rope_in_attention(q, k, v, kc, meta)
        if fused:
            out = ops.rope_attention(q, k, v, meta.positions, cos_sin, slots,
                                     kc, vc, meta, D ** -0.5)
        else:
            ops.rope_kv_append(q, k, v, meta.positions, cos_sin, slots, kc, vc)
            out = ops.attention(q, k, v, kc, vc, meta, D ** -0.5)
        outs.append(out.float())
        pages.append([c.view(torch.uint8) for c in (kc, vc)])
    assert all(torch.equal(a, b) for a, b in zip(*pages))
    assert (outs[0] - outs[1]).abs().max() <= 2.0 ** -8 * outs[1].abs().max()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("rows,kv,groups,shared", [
    (2, 1, 1, 16), (3, 2, 1, 32), (5, 2, 2, 48), (17, 1, 16, 96), (18, 1, 18, 512),
    (33, 2, 17, 80), (40, 8, 3, 176), (8, 1, 1, 1600)])
def test_pages_of_shared_prompts(rows, kv, groups, shared, fp8):
    """Rows that begin with the same pages, one after the other or at a distance,
    some as long as those, against copies of the pages for every row: same bits."""
    g = torch.Generator().manual_seed(rows)
    group, kind = 4, torch.float8_e4m3fn if fp8 else torch.bfloat16
    heads, first = group * kv, shared // 16
    lens = torch.randint(shared + 1, shared + 150, (rows,), generator=g)
    lens[rows // 2:rows // 2 + 2] = shared + 1
    own = -(-lens // 16) - first
    total = groups * first + int(own.sum())
    caches = [torch.randn(total, kv, 16, D, generator=g).to(kind)
              for _ in range(2)]
    order = torch.randperm(total, generator=g).int()
    bt = torch.zeros(rows, first + int(own.max()) + 1, dtype=torch.int32)
    at = groups * first
    for i in range(rows):
        bt[i, :first] = order[i % groups * first:][:first]
        bt[i, first:first + own[i]] = order[at:at + own[i]]
        at += int(own[i])
    each = torch.arange(bt.numel(), dtype=torch.int32).view_as(bt)
    cos_sin = torch.randn(2000, D, generator=g).to(DEV)
    qkv = torch.randn(rows, heads + 2 * kv, D, generator=g).bfloat16().to(DEV)
    outs, pages = [], []
    for table, kept in ((bt, caches),
                        (each, [c[bt.flatten().long()] for c in caches])):
        last = table.gather(1, (lens - 1).div(16, rounding_mode="floor")[:, None])
        slots = (last[:, 0].long() * 16 + (lens - 1) % 16).to(DEV)
        meta = ForwardMeta("decode", (lens - 1).to(DEV), slots,
                           block_tables=table.to(DEV),
                           seq_lens=lens.int().to(DEV))
        kc, vc = (c.clone().to(DEV) for c in kept)
        q, k, v = qkv.clone().split([heads, kv, kv], 1)
        assert ops._rope_in_attention(q, k, v, kc, meta)
        outs.append(ops.rope_attention(q, k, v, meta.positions, cos_sin, slots,
                                       kc, vc, meta, D ** -0.5))
        pages.append([c.view(torch.uint8)[last[:, 0].long().to(DEV)]
                      for c in (kc, vc)])
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(*outs)
    assert all(torch.equal(a, b) for a, b in zip(*pages))


@pytest.mark.parametrize("parts", [2, 15, 16, 17, 33, 64])
def test_parts_of_decode_attention(parts):
    """More parts than one has 32 tokens for, and than are loaded at a time."""
    g = torch.Generator().manual_seed(parts)
    lens, kv, group = [1, 700, 4001], 2, 4
    tables = [-(-x // 16) for x in lens]
    caches = [torch.randn(sum(tables), kv, 16, D, generator=g).bfloat16()
              for _ in range(2)]
    order = torch.randperm(sum(tables), generator=g).int().split(tables)
    bt = torch.zeros(3, max(tables), dtype=torch.int32)
    for row, pages in zip(bt, order):
        row[:len(pages)] = pages
    q = torch.randn(3, kv * group, D, generator=g).bfloat16().to(DEV)
    out = torch.empty_like(q)
    ws = torch.full((3 * kv * group * parts * (D + 2),), float("nan"),
                    device=DEV)
    ops._native().paged_attn(
        out, q, *(c.to(DEV) for c in caches), bt.to(DEV),
        torch.tensor(lens, dtype=torch.int32, device=DEV), None, D ** -0.5,
        ws, parts)
    for i, n in enumerate(lens):
        k, v = (c[order[i].long()].float().transpose(1, 2).reshape(-1, kv, D)
                [:n] for c in caches)
        _check(out[i:i + 1], _reference(q[i:i + 1], k, v, n - 1, D ** -0.5),
               2.0 ** -14)


@pytest.mark.parametrize("rows", [8, 103, 104])    # by rows, and in tiles
def test_weights_over_bf16_pages_are_floats(rows):
    """Values that cancel: what is left is the error of the weights.

    Scores of at most one are off by a few 2^-24 and their exponentials by
    about 2^-23; three bf16 parts hold a weight to 2^-25 and two to 2^-18."""
    g = torch.Generator().manual_seed(8)
    before, total = 64, 64 + rows
    q = (torch.randn(D, generator=g) * 0.3).bfloat16()
    k = (torch.randn(total, D, generator=g) * 0.3).bfloat16()
    scale = D ** -0.5
    w = (k[:before].double() @ q.double() * scale).exp()
    v = torch.randn(before, D, generator=g).bfloat16()
    for t in range(before - 4, before):         # each takes 2^-9 of the rest
        v[t:] = 0
        v[t] = (-(w @ v.double()) / w[t]).bfloat16()
    # the portion's own tokens add nothing
    v = torch.cat([v, torch.zeros(rows, D).bfloat16()])
    pages = total // 16 + (total % 16 > 0)
    kc, vc = (torch.zeros(pages * 16, 1, D).bfloat16() for _ in range(2))
    kc[:total, 0], vc[:total, 0] = k, v
    kc, vc = (c.view(pages, 16, 1, D).transpose(1, 2).contiguous().to(DEV)
              for c in (kc, vc))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    meta = ForwardMeta("prefill", None, None, seq_start=i32([0, rows]),
                       row_seq=i32([0] * rows),
                       ctx_lens=i32(list(range(before + 1, total + 1))),
                       block_tables=i32([list(range(pages))]),
                       fresh_prefill=False)
    out = ops.attention(q.expand(rows, 1, D).contiguous().to(DEV), None, None,
                        kc, vc, meta, scale)
    size = (w[:, None] * v[:before].double().abs()).sum(0) / w.sum()
    assert (out[:, 0].double().cpu().abs() <= 2.0 ** -21 * size).all()


def _pages_of(lens, kv, fp8, g):
    """(k, v of every sequence in order, the pages with NaN after each one's
    last token, block tables)"""
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    tables = [-(-n // 16) for n in lens]
    order = torch.randperm(sum(tables), generator=g).split(tables)
    bt = torch.zeros(len(lens), max(tables) + 1, dtype=torch.int32)
    both = [[torch.randn(n, kv, D, generator=g).to(kind).float() for n in lens]
            for _ in range(2)]
    caches = []
    for rows in both:
        cache = torch.full((sum(tables), kv, 16, D), float("nan"))
        for i, pages in enumerate(order):
            bt[i, :tables[i]] = pages
            whole = torch.full((tables[i] * 16, kv, D), float("nan"))
            whole[:lens[i]] = rows[i]
            cache[pages] = whole.view(-1, 16, kv, D).transpose(1, 2)
        caches.append(cache.to(kind).to(DEV))
    return both, caches, bt


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("split", [1, 3])
def test_nan_after_the_last_token_in_decode(split, fp8):
    from hyperspot import _C
    g = torch.Generator().manual_seed(9)
    lens, kv, heads = [1, 15, 17, 31, 33, 50, 64, 130, 400], 2, 8
    (k, v), (kc, vc), bt = _pages_of(lens, kv, fp8, g)
    q = torch.randn(len(lens), heads, D, generator=g).bfloat16().to(DEV)
    out = torch.empty_like(q)
    ws = torch.empty(len(lens) * heads * split * (D + 2), device=DEV) \
        if split > 1 else None
    _C.paged_attn(out, q, kc, vc, bt.to(DEV),
                  torch.tensor(lens, dtype=torch.int32, device=DEV), None,
                  D ** -0.5, ws, split)
    for i, n in enumerate(lens):
        _check(out[i:i + 1], _reference(q[i:i + 1], k[i], v[i], n - 1,
                                        D ** -0.5), 2.0 ** -14)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("portions", [
    [(5, 90), (40, 17), (64, 3), (30, 33)], [(100, 130)], [(1, 103)],
    [(1, 104)],
])
def test_nan_after_the_last_token_of_portions(portions, fp8):
    g = torch.Generator().manual_seed(10)
    kv, heads = 2, 8
    lens, rows = [b + n for b, n in portions], [n for _, n in portions]
    (k, v), (kc, vc), bt = _pages_of(lens, kv, fp8, g)
    q = torch.randn(sum(rows), heads, D, generator=g).bfloat16().to(DEV)
    starts = [sum(rows[:i]) for i in range(len(rows) + 1)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    meta = ForwardMeta("prefill", None, None, seq_start=i32(starts),
                       row_seq=i32([i for i, n in enumerate(rows)
                                    for _ in range(n)]),
                       ctx_lens=i32([c + 1 for b, n in portions
                                     for c in range(b, b + n)]),
                       block_tables=bt.to(DEV), fresh_prefill=False)
    out = ops.attention(q, None, None, kc, vc, meta, D ** -0.5)
    for i, (b, n) in enumerate(portions):
        at = slice(starts[i], starts[i + 1])
        _check(out[at], _reference(q[at], k[i], v[i], b, D ** -0.5),
               2.0 ** -14)


@pytest.mark.parametrize("shift", [0, 4])      # elements: pages off 16 bytes
def test_portions_with_longer_tables(shift):
    """What the row-by-row kernel takes."""
    g = torch.Generator().manual_seed(11)
    kv, heads, before, n = 2, 8, 40, 120
    (k, v), caches, bt = _pages_of([before + n], kv, False, g)
    kc, vc = (torch.cat([c.new_zeros(shift), c.view(-1)])[shift:].view_as(c)
              for c in caches)
    q = torch.randn(n, heads, D, generator=g).bfloat16().to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    meta = ForwardMeta("prefill", None, None, seq_start=i32([0, n]),
                       row_seq=i32([0] * (n + 7)),
                       ctx_lens=i32(list(range(before + 1, before + n + 8))),
                       block_tables=bt.to(DEV), fresh_prefill=False)
    out = ops.attention(q, None, None, kc, vc, meta, D ** -0.5)
    _check(out, _reference(q, k[0], v[0], before, D ** -0.5), 2.0 ** -14)
