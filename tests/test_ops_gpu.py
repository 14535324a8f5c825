"""GPU numerics tests: every gfx950 HIP kernel vs the plain-PyTorch fp32
reference of the same op (hyperspot.ops.torch_ref).  bf16 I/O tolerances."""

import pytest
import torch

import hyperspot.ops as ops
from hyperspot.ops import torch_ref as R

pytestmark = pytest.mark.gpu

DEV = "cuda"


def setup_module():
    assert ops.have_native(), \
        "hyperspot._C must be built on GPU boxes (python csrc/build.py)"


def _randn_bf16(*shape, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).bfloat16().to(DEV)


@pytest.mark.parametrize("hidden", [2048, 4096, 8192])
def test_rmsnorm(hidden):
    x = _randn_bf16(33, hidden)
    w = _randn_bf16(hidden, seed=1)
    out = ops.rmsnorm(x, w, 1e-5)
    ref = R.rmsnorm(x.float().cpu(), w.float().cpu(), 1e-5)
    assert torch.allclose(out.float().cpu(), ref, atol=3e-2, rtol=3e-2)


def test_fused_add_rmsnorm():
    x = _randn_bf16(17, 4096)
    res = _randn_bf16(17, 4096, seed=2)
    w = _randn_bf16(4096, seed=3)
    x_ref, res_ref = x.float().cpu(), res.float().cpu()
    out, new_res = ops.fused_add_rmsnorm(x, res, w, 1e-5)
    ref_out, ref_res = R.fused_add_rmsnorm(x_ref, res_ref,
                                           w.float().cpu(), 1e-5)
    assert torch.allclose(new_res.float().cpu(), ref_res, atol=3e-2, rtol=3e-2)
    assert torch.allclose(out.float().cpu(), ref_out, atol=4e-2, rtol=4e-2)


def test_rope_kv_append():
    T, H, KV, D, BS, NB = 9, 8, 2, 128, 16, 8
    q = _randn_bf16(T, H, D)
    k = _randn_bf16(T, KV, D, seed=1)
    v = _randn_bf16(T, KV, D, seed=2)
    pos = torch.tensor([0, 1, 2, 5, 9, 100, 101, 4, 7], device=DEV)
    slots = torch.tensor([0, 1, 2, 17, 18, 33, 40, -1, 55], device=DEV)
    cos_sin = R.rope_cos_sin(torch.arange(256), D, 500000.0).to(DEV)
    k_cache = torch.zeros(NB, KV, BS, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.zeros_like(k_cache)
    q_ref, k_ref = R.apply_rope(q.float().cpu(), k.float().cpu(),
                                pos.cpu(), 500000.0)
    ops.rope_kv_append(q, k, v, pos, cos_sin, slots, k_cache, v_cache)
    assert torch.allclose(q.float().cpu(), q_ref, atol=3e-2, rtol=3e-2)
    assert torch.allclose(k.float().cpu(), k_ref, atol=3e-2, rtol=3e-2)
    # cache contents (skip slot -1 row)
    kc_ref = torch.zeros(NB, KV, BS, D)
    vc_ref = torch.zeros(NB, KV, BS, D)
    mask = slots.cpu() >= 0
    R.kv_cache_append(k.float().cpu()[mask], v.float().cpu()[mask],
                      kc_ref, vc_ref, slots.cpu()[mask])
    assert torch.allclose(k_cache.float().cpu(), kc_ref, atol=3e-2, rtol=3e-2)
    assert torch.allclose(v_cache.float().cpu(), vc_ref, atol=3e-2, rtol=3e-2)
    # slot -1 must not be written anywhere: caches zero outside ref slots
    untouched = torch.ones(NB * BS, dtype=torch.bool)
    untouched[slots.cpu()[mask]] = False
    kc = k_cache.float().cpu().permute(0, 2, 1, 3).reshape(NB * BS, KV, D)
    assert (kc[untouched] == 0).all()


@pytest.mark.parametrize("heads,kv,dim,fp8", [
    (8, 2, 128, False), (1, 1, 128, True), (32, 8, 128, True), (28, 4, 128, False),
    (5, 3, 64, False)])
def test_rope_kv_append_of_any_stride(heads, kv, dim, fp8):
    """Rows 16 bytes apart or not, the same bits; one whose slot is negative."""
    T, BS, NB = 37, 16, 5
    g = torch.Generator().manual_seed(heads)
    x = torch.randn(T, heads + 2 * kv, dim, generator=g).bfloat16().to(DEV)
    pos = torch.randint(0, 256, (T,), generator=g).to(DEV)
    slots = (torch.randperm(NB * BS, generator=g)[:T]).to(DEV)
    slots[5] = -1
    cos_sin = R.rope_cos_sin(torch.arange(256), dim, 500000.0).to(DEV)
    got = []
    for gap in (0, 4):                      # elements between two rows of q, k
        caches = [torch.zeros(NB, kv, BS, dim, device=DEV).to(
            torch.float8_e4m3fn if fp8 else torch.bfloat16) for _ in "kv"]
        parts = [torch.zeros(T, n * dim + gap, device=DEV).bfloat16()
                 for n in (heads, kv)]
        q, k = (p[:, :n * dim].unflatten(1, (n, dim))
                for p, n in zip(parts, (heads, kv)))
        q.copy_(x[:, :heads])
        k.copy_(x[:, heads:heads + kv])
        v = x[:, heads + kv:].contiguous()
        ops.rope_kv_append(q, k, v, pos, cos_sin, slots, *caches)
        assert all((p[:, -gap:] == 0).all() for p in parts if gap)
        got.append([t.contiguous().view(torch.uint8)
                    for t in (q, k, *caches)])
    for a, b in zip(*got):
        assert torch.equal(a, b)
    cos, sin = cos_sin[pos].double().chunk(2, -1)
    want = R._rotate_neox(x[:, :heads].double(), cos, sin)
    out = got[0][0].view(torch.bfloat16).view(want.shape).double()
    # rounded once
    assert ((out - want).abs() <= want.abs() * 2.0 ** -8 + 1e-6).all()
    rows = caches[1].float().transpose(1, 2).reshape(NB * BS, kv, dim)
    kept = slots >= 0
    assert torch.equal(rows[slots[kept]],
                       x[:, heads + kv:][kept].to(caches[1].dtype).float())
    rows[slots[kept]] = 0
    assert (rows == 0).all()


@pytest.mark.parametrize("group,heads_kv", [(4, 8), (8, 1), (1, 2)])
def test_paged_attn_decode(group, heads_kv):
    torch.manual_seed(0)
    B, D, BS, NB = 5, 128, 16, 64
    H = group * heads_kv
    maxb = 8
    q = _randn_bf16(B, H, D)
    k_cache = _randn_bf16(NB, heads_kv, BS, D, seed=1)
    v_cache = _randn_bf16(NB, heads_kv, BS, D, seed=2)
    bt = torch.randperm(NB, device=DEV, dtype=torch.int32)[: B * maxb] \
        .reshape(B, maxb).contiguous()
    seq_lens = torch.tensor([1, 16, 17, 100, 128], dtype=torch.int32,
                            device=DEV)
    out = ops.paged_attn_decode(q, k_cache, v_cache, bt, seq_lens,
                                D ** -0.5)
    ref = R.paged_attn_decode(q.float().cpu(), k_cache.float().cpu(),
                              v_cache.float().cpu(), bt.cpu(),
                              seq_lens.cpu(), D ** -0.5)
    assert torch.allclose(out.float().cpu(), ref, atol=2e-2, rtol=2e-2)


def test_paged_attn_prefill_matches_varlen_ref():
    """Prefill through the cache == varlen causal attention."""
    torch.manual_seed(0)
    H, KV, D, BS = 4, 2, 128, 16
    lens = [33, 7, 64]
    T = sum(lens)
    NB = 32
    q = _randn_bf16(T, H, D)
    k = _randn_bf16(T, KV, D, seed=1)
    v = _randn_bf16(T, KV, D, seed=2)
    k_cache = torch.zeros(NB, KV, BS, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.zeros_like(k_cache)
    # identity-ish paging: seq i gets consecutive blocks
    tables, slots, row_seq, ctx = [], [], [], []
    next_blk = 0
    for si, n in enumerate(lens):
        nb = (n + BS - 1) // BS
        blocks = list(range(next_blk, next_blk + nb))
        next_blk += nb
        tables.append(blocks + [0] * (8 - nb))
        for p in range(n):
            slots.append(blocks[p // BS] * BS + p % BS)
            row_seq.append(si)
            ctx.append(p + 1)
    slots_t = torch.tensor(slots, device=DEV)
    R.kv_cache_append(k.float().cpu(), v.float().cpu(),
                      kc := torch.zeros(NB, KV, BS, D),
                      vc := torch.zeros(NB, KV, BS, D), slots_t.cpu())
    k_cache.copy_(kc.bfloat16())
    v_cache.copy_(vc.bfloat16())
    bt = torch.tensor(tables, dtype=torch.int32, device=DEV)
    out = torch.empty_like(q)
    from hyperspot import _C
    _C.paged_attn(out, q, k_cache, v_cache, bt,
                  torch.tensor(ctx, dtype=torch.int32, device=DEV),
                  torch.tensor(row_seq, dtype=torch.int32, device=DEV),
                  D ** -0.5, None, 1)
    ss = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32)
    ref = R.prefill_attn(q.float().cpu(), k.float().cpu(), v.float().cpu(),
                         ss, D ** -0.5)
    assert torch.allclose(out.float().cpu(), ref, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("lens,H,KV", [
    ([5, 300, 64], 8, 2),     # partial tiles + >256-row tile crossing
    ([513], 4, 4),            # MHA, 3 q tiles
    ([33, 16], 8, 1),         # group=8
])
def test_attn_prefill_mfma_vs_ref(lens, H, KV):
    torch.manual_seed(1)
    D = 128
    T = sum(lens)
    q = _randn_bf16(T, H, D, seed=11)
    k = _randn_bf16(T, KV, D, seed=12)
    v = _randn_bf16(T, KV, D, seed=13)
    ss = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=DEV)
    out = torch.empty_like(q)
    from hyperspot import _C
    _C.attn_prefill_mfma(out, q, k, v, ss, max(lens), D ** -0.5)
    ref = R.prefill_attn(q.float().cpu(), k.float().cpu(), v.float().cpu(),
                         ss.cpu(), D ** -0.5)
    assert torch.allclose(out.float().cpu(), ref, atol=2.5e-2, rtol=2.5e-2)


def test_attn_prefill_mfma_strided_views():
    """Exercise the fused-qkv strided-view path end to end."""
    torch.manual_seed(2)
    H, KV, D = 4, 2, 128
    lens = [40, 17]
    T = sum(lens)
    qkv = _randn_bf16(T, (H + 2 * KV) * D, seed=21)
    q = qkv[:, :H * D].view(T, H, D)
    k = qkv[:, H * D:(H + KV) * D].view(T, KV, D)
    v = qkv[:, (H + KV) * D:].view(T, KV, D)
    ss = torch.tensor([0, 40, 57], dtype=torch.int32, device=DEV)
    out = torch.empty(T, H, D, dtype=torch.bfloat16, device=DEV)
    from hyperspot import _C
    _C.attn_prefill_mfma(out, q, k, v, ss, 40, D ** -0.5)
    ref = R.prefill_attn(q.float().cpu(), k.float().cpu(), v.float().cpu(),
                         ss.cpu(), D ** -0.5)
    assert torch.allclose(out.float().cpu(), ref, atol=2.5e-2, rtol=2.5e-2)


@pytest.mark.gpu
def test_attn_prefill_mfma_rows_far_apart():
    """Rows of keys and values that 32 bits of offset do not reach."""
    far = 1 << 25
    qkv = torch.randn(70, 4, 128, device=DEV, dtype=torch.bfloat16)
    wide = torch.empty(69 * far + 256, device=DEV, dtype=torch.bfloat16)
    k, v = (wide[i * 128:].as_strided((70, 1, 128), (far, 128, 1))
            for i in range(2))
    k.copy_(qkv[:, :1])
    v.copy_(qkv[:, 1:2])
    start = torch.tensor([0, 70], dtype=torch.int32, device=DEV)
    outs = []
    for kv in ((k, v), (k.contiguous(), v.contiguous())):
        out = torch.empty(70, 2, 128, device=DEV, dtype=torch.bfloat16)
        ops._native().attn_prefill_mfma(out, qkv[:, 2:], *kv, start, 70, 0.09)
        outs.append(out)
    assert torch.equal(*outs)



def test_silu_mul():
    x = _randn_bf16(65, 2 * 1024)
    out = ops.silu_mul(x)
    ref = R.silu_mul(x.float().cpu())
    assert torch.allclose(out.float().cpu(), ref, atol=2e-2, rtol=2e-2)


def test_silu_mul_of_many_rows():
    """Beyond 40 M outputs its loads are others; a row's bits are not."""
    rows, inter = 2999, 13992
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(rows, 2 * inter, generator=g, device=DEV).bfloat16()
    assert rows * inter >= 40 << 20
    out = ops.silu_mul(x)
    for a in range(0, rows, 1000):
        assert torch.equal(out[a:a + 1000], ops.silu_mul(x[a:a + 1000]))


def test_greedy_sample():
    torch.manual_seed(0)
    logits = _randn_bf16(64, 128256)
    out = ops.greedy_sample(logits)
    # ties are possible in bf16: check the VALUE is the max
    mx = logits.float().max(-1).values
    picked = logits.float().gather(1, out[:, None].to(DEV)).squeeze(1)
    assert torch.equal(picked.cpu(), mx.cpu())


def test_inv_cdf_sample_matches_reference():
    torch.manual_seed(0)
    B, V = 16, 128256
    logits = torch.randn(B, V, device=DEV)
    u = torch.rand(B, device=DEV)
    ones = torch.ones(B, device=DEV)
    out = ops.sample(logits, ones, ones,
                     torch.zeros(B, dtype=torch.int32, device=DEV), u)
    ref = R.sample(logits.cpu(), torch.ones(B), torch.ones(B),
                   torch.zeros(B, dtype=torch.int32), u.cpu())
    # fp-association differences can shift the crossing by a hair when u
    # lands exactly on a boundary; require >= 15/16 exact matches and
    # adjacent-index otherwise
    same = (out.cpu() == ref).sum().item()
    assert same >= B - 1, (out.cpu(), ref)


def test_sample_dispatch_topk_topp_gpu():
    torch.manual_seed(0)
    B, V = 8, 1000
    logits = _randn_bf16(B, V).float()
    topk = logits.topk(5, dim=-1).indices.cpu()
    for trial in range(5):
        t = ops.sample(logits, torch.ones(B, device=DEV),
                       torch.ones(B, device=DEV),
                       torch.full((B,), 5, dtype=torch.int32, device=DEV),
                       torch.rand(B, device=DEV))
        for b in range(B):
            assert t[b].cpu() in topk[b]


@pytest.mark.gpu
def test_moe_grouped_ffn_matches_ref():
    """Grouped MFMA expert GEMMs + combine vs the per-expert loop."""
    import hyperspot.ops as ops
    torch.manual_seed(0)
    dev = "cuda:0"
    T, H, I, E, K = 96, 256, 256, 4, 2
    x = (torch.randn(T, H, device=dev) * 0.3).to(torch.bfloat16)
    w13 = (torch.randn(E, 2 * I, H, device=dev) * 0.05).to(torch.bfloat16)
    w2 = (torch.randn(E, H, I, device=dev) * 0.05).to(torch.bfloat16)
    logits = torch.randn(T, E, device=dev)
    w, ids = logits.softmax(-1).topk(K, dim=-1)
    w = (w / w.sum(-1, keepdim=True)).float()

    out = ops.moe_ffn(x, w13, w2, w, ids.to(torch.int32))

    ref = torch.zeros(T, H, device=dev, dtype=torch.float32)
    xf = x.float()
    for t in range(T):
        for k in range(K):
            e = int(ids[t, k])
            gu = xf[t] @ w13[e].float().t()
            g, u = gu[:I], gu[I:]
            y = (g * torch.sigmoid(g) * u) @ w2[e].float().t()
            ref[t] += w[t, k] * y
    err = (out.float() - ref).abs().max().item()
    scale = ref.abs().max().item()
    assert err < 0.02 * scale + 0.02, (err, scale)


@pytest.mark.gpu
@pytest.mark.parametrize("segments", [1, 2, 4])
def test_moe_splitk_matches_single_segment(segments):
    """The grouped GEMM whose K may be split (fp32 partials + reduce), with
    every degree that 12 k-chunks allow, against float64 on the same sorted
    choices.  Bound: the result is rounded to bf16 (2^-9 of it), and sums of K
    products are off by K 2^-24 of the sum of their sizes."""
    import hyperspot.ops as ops
    from hyperspot import _C
    torch.manual_seed(1)
    dev = "cuda:0"
    T, N, K, E, top = 160, 256, 768, 4, 2
    x = (torch.randn(T, K, device=dev) * 0.3).to(torch.bfloat16)
    w = (torch.randn(E, N, K, device=dev) * 0.04).to(torch.bfloat16)
    ids = torch.randn(T, E, device=dev).topk(top, dim=-1).indices.int()
    order, expert, place = ops._moe_sort(ids, E, N, K, ops.MOE_BM)
    out = torch.full((order.numel(), N), float("nan"), dtype=torch.bfloat16,
                     device=dev)
    ws = torch.full((segments * out.numel(),), float("nan"), device=dev) \
        if segments > 1 else None
    _C.moe_gemm(out, x, w, order, expert, top, segments, ws)
    xd, wd = x.double().cpu(), w.double().cpu()
    got = out[place.long().view(-1)].double().cpu()
    for c, e in enumerate(ids.view(-1).tolist()):
        ref, size = wd[e] @ xd[c // top], wd[e].abs() @ xd[c // top].abs()
        assert ((got[c] - ref).abs()
                <= ref.abs() * 2.0 ** -8 + size * K * 2.0 ** -24).all()


@pytest.mark.gpu
def test_moe_splitk_degree(monkeypatch):
    """The degree that is chosen, and HS_MOE_SPLITK, which forces it."""
    import hyperspot.ops as ops
    degree = lambda *a: ops._moe_splitk(*a, 64, "cuda:0")[0]
    assert [degree(n, 12) for n in (12, 600, 1024)] == [4, 2, 1]
    for forced in (1, 2, 4):
        monkeypatch.setenv("HS_MOE_SPLITK", str(forced))
        assert degree(12, 12) == forced and degree(1024, 12) == 1
