"""e4m3 products in tiles and in parts of K, against float64.

Bound: the result is rounded to bf16 (2^-9 of it) and sums K products of float
precision in any order (K 2^-24 of the sum of their sizes)."""

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops

DEV = "cuda:0"
E4M3 = torch.float8_e4m3fn


def _operands(M, N, K, pad=0):
    g = torch.Generator().manual_seed(M + N)
    new = lambda r: torch.randn(r, K + pad, generator=g).to(E4M3).to(DEV)[:, pad:]
    scale = lambda r: (torch.rand(r, generator=g) + 0.5).to(DEV)
    return ops.QTensor(new(M), scale(M)), new(N), scale(N)


def _check(out, q, w, ws):
    x, w = q.data.double().cpu(), w.double().cpu()
    s = q.scale.double().cpu()[:, None] * ws.double().cpu()
    ref = (x @ w.t()) * s
    bound = ref.abs() * 2.0 ** -8 \
        + x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().t()) * s
    assert ((out.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", [(64, 32), (64, 64), (64, 128)])
@pytest.mark.parametrize("M,N,K,parts", [
    (1, 4, 256, 1), (31, 60, 512, 2), (64, 64, 768, 3), (65, 132, 1280, 4),
    (128, 64, 2048, 8), (129, 260, 2304, 8), (33, 1028, 1792, 7),
    (64, 4100, 512, 2), (128, 8200, 256, 1),
])
def test_gemm(M, N, K, parts, bm, bn):
    q, w, ws = _operands(M, N, K, 16)       # rows are views into wider ones
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    part = torch.full((parts, M, N), float("nan"), device=DEV)
    ops._native().gemm_split(out, q.data, w, part, bm, bn, parts, q.scale, ws)
    _check(out, q, w, ws)
    if parts > 1:
        part.fill_(float("nan"))
        ops._native().gemm_split(None, q.data, w, part, bm, bn, parts, q.scale,
                                 ws)
        _check(part.sum(0), q, w, ws)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (1, 4, 16), (3, 20, 528), (16, 260, 1040), (17, 2052, 2048), (32, 4100, 272),
    (33, 516, 2064), (64, 12, 1024), (8, 6144, 4096), (1, 36, 28672)])
def test_products_of_few_rows(M, N, K):
    """Columns that end within a line or a load, outputs within a tile."""
    q, w, ws = _operands(M, N, K, 16)       # rows are views into wider ones
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops._native().gemm_rows(out, q.data, w, q.scale, ws)
    _check(out, q, w, ws)
    with pytest.raises(RuntimeError):
        ops._native().gemm_rows(out, q.data, w, q.scale)


def test_rule_of_few_rows():
    for M, N, K, parts, rule in [
            (1, 6144, 4096, False, True), (32, 6144, 4096, False, True),
            (33, 6144, 4096, False, False), (1, 4096, 4096, True, False),
            (16, 2048, 7168, False, True), (17, 2048, 7168, False, True),
            (16, 4096, 14336, False, False), (1, 4096, 14336, True, False),
            (1, 28672, 4096, False, False), (8, 8880, 14592, False, True),
            (0, 4096, 4096, False, False), (1, 4098, 4096, False, False),
            (1, 4096, 4104, False, False), (1, 64, 1024, False, False),
            (1, (1 << 24) - 4, 16, False, True), (1, 1 << 24, 16, False, False),
            (32, 1 << 31, 16, False, False)]:
        assert ops._rows_q_sizes(M, N, K, parts) == rule, (M, N, K, parts)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 64, 65, 128, 129])
@pytest.mark.parametrize("N,K", [(4096, 4096), (2048, 7168), (12288, 1024),
                                 (3600, 5120), (2048, 2048), (4096, 14336),
                                 (20480, 2048)])
@pytest.mark.parametrize("parts", [False, True])
def test_linear_q(M, N, K, parts):
    q, w, ws = _operands(M, N, K)
    out = ops.linear_q(q, w, ws, parts)
    rule = ops._tiles_q(M, N, K, parts)
    assert (rule is None) == (M == 129 or ops._tiled_q(q, w, ws, parts) is None)
    assert isinstance(out, ops.Parts) == (
        parts and rule is not None and rule[2] > 1 and N <= 8192)
    _check(out.data.sum(0) if isinstance(out, ops.Parts) else out, q, w, ws)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,hidden,parts", [
    (1, 8, 2), (3, 2048, 8), (64, 2056, 5), (17, 4096, 4), (5, 8192, 3)])
def test_parts_add_norm(rows, hidden, parts):
    """As the sum rounded to bf16, then the add and norm."""
    g = torch.Generator().manual_seed(rows)
    p = torch.randn(parts, rows, hidden, generator=g).to(DEV)
    res = torch.randn(rows, hidden, generator=g).bfloat16().to(DEV)
    w = torch.rand(hidden, generator=g).bfloat16().to(DEV)
    y = p[0].clone()
    for z in range(1, parts):
        y += p[z]
    want, want_res = ops.fused_add_rmsnorm_q(y.bfloat16(), res.clone(), w, 1e-5)
    got, got_res = ops.fused_add_rmsnorm_q(ops.Parts(p), res, w, 1e-5)
    assert torch.equal(got_res, want_res)
    # the sums of squares are in another order: the last bit of a scale
    torch.testing.assert_close(got.scale, want.scale, rtol=1e-6, atol=0)
    a, b = got.data.float() * got.scale[:, None], \
        want.data.float() * want.scale[:, None]
    # a value between two steps of e4m3 may take the other one
    assert ((a - b).abs() <= b.abs() * 0.13 + want.scale[:, None] * 2e-3).all()
    assert (a != b).float().mean() <= 0.01 or rows * hidden < 1000


def test_rule_stays_in_what_the_kernel_takes():
    taken = 0
    for M in (*range(1, 130, 7), 64, 65, 128):
        for N in (4, 512, 1000, 2048, 3600, 4096, 6144, 8200, 28672, 1 << 17):
            for K in (256, 1024, 2048, 4096, 5120, 7168, 8192, 14336, 1 << 16):
                for parts in (False, True):
                    rule = ops._tiles_q(M, N, K, parts)
                    if rule is None:
                        continue
                    taken += 1
                    bm, bn, z = rule
                    assert (bm, bn) in ((64, 32), (64, 64), (64, 128))
                    assert 1 <= z <= min(8, K // 256)
    assert taken > 100
    assert ops._tiles_q(64, 4096, 4096 + 128, False) is None
    assert ops._tiles_q(129, 4096, 4096, False) is None
