"""Products of many rows in tiles of 128 to 256 rows, against float64, at the edges
of tiles, and the rules that choose them.

Bounds: products are exact in float and summed in float, 2^-22 of the sum of
magnitudes; results are rounded to bf16, half a step is at most 2^-8 of them."""

import random

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops

DEV = "cuda:0"


def _inputs(M, N, K, pad=0):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + pad, generator=g).bfloat16().to(DEV)[:, :K]
    w = (torch.randn(N, K + pad, generator=g) * K ** -0.5).bfloat16()
    return x, w.to(DEV)[:, :K]


def _bounds(x, w):
    x, w = x.double(), w.double()
    return x @ w.t(), x.abs() @ w.abs().t() * 2.0 ** -22


@pytest.mark.gpu
@pytest.mark.parametrize("high", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("bn", [128, 256])
@pytest.mark.parametrize("M,N,K,pad", [
    (1, 8, 64, 0), (-1, 264, 128, 8), (0, 256, 192, 0), (1, 520, 320, 64),
    (700, 1032, 448, 0)])
def test_tiles(high, bn, M, N, K, pad):
    """M: rows beside a whole number of tiles, or some tiles of rows and nine of
    them, more than go together."""
    M = 9 * 32 * high + 5 if M == 700 else 32 * high + M
    x, w = _inputs(M, N, K, pad)
    want, slack = _bounds(x, w)
    out = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._native().gemm_wide(out, x, w, None, high, bn)
    assert ((out.double() - want).abs()
            <= 2.0 ** -8 * want.abs() + 1.01 * slack).all()
    for parts in {2, K // 64} - {1}:
        if parts > K // 64 or parts > 8:
            continue
        part = torch.full((parts, M, N), 7.0, device=DEV)
        ops._native().gemm_wide(None, x, w, part, high, bn, parts)
        edge = [K // 64 * z // parts * 64 for z in range(parts + 1)]
        for z in range(parts):
            p, s = _bounds(x[:, edge[z]:edge[z + 1]], w[:, edge[z]:edge[z + 1]])
            assert ((part[z].double() - p).abs() <= s).all()


@pytest.mark.gpu
@pytest.mark.parametrize("high", [4, 5, 8])
@pytest.mark.parametrize("bn", [128, 256])
@pytest.mark.parametrize("N,K", [(16, 64), (272, 128), (784, 320)])
def test_gated_tiles(high, bn, N, K):
    M = 32 * high * 2 - 7
    x, w = _inputs(M, N, K)
    out = torch.full((M, N // 2), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._native().gemm_wide(out, x, w, None, high, bn, gated=True)
    (gate, up), (dg, du) = (t.chunk(2, -1) for t in _bounds(x, w))
    want = torch.nn.functional.silu(gate) * up
    # |silu'| <= 1.1, |silu(g)| <= |g|; the exponential's error is 2^-20
    slack = 1.1 * dg * up.abs() + gate.abs() * du + 2.0 ** -20 * want.abs()
    assert ((out.double() - want).abs()
            <= 2.0 ** -8 * want.abs() + 1.01 * slack).all()


@pytest.mark.gpu
def test_numbers_that_are_not_finite():
    """They stay in their rows, and rows past the end do not matter."""
    x, w = _inputs(300, 264, 192)
    x[7, 3], x[299, 191], w[5, 0] = float("nan"), float("inf"), float("inf")
    out = torch.empty(300, 264, dtype=torch.bfloat16, device=DEV)
    ops._native().gemm_wide(out, x, w, None, 5, 128)
    want = x.float() @ w.float().t()
    assert torch.equal(out.isfinite(), want.isfinite())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (257, 4096, 14336), (600, 4096, 10240), (513, 2048, 7168),
    (1400, 4096, 10240), (129, 4096, 14336), (256, 4096, 10240)])
def test_parts_and_norm(M, N, K):
    assert ops._wide_parts(M, N, K) and not ops._wide_parts(128, N, K)
    x, w = _inputs(M, N, K)
    got = ops.linear_parts(x, w)
    parts = ops._wide_parts(M, N, K)[2]
    assert isinstance(got, ops.Parts) and got.data.shape == (parts, M, N)
    want, slack = _bounds(x, w)
    y = got.data.sum(0)
    assert ((y.double() - want).abs()
            <= 2.0 ** -8 * want.abs() + 2 * slack).all()
    # the norms add the parts in their order and round the sum as a product is
    g = torch.Generator().manual_seed(M)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().to(DEV)
    res, norm, router = rand(M, N), rand(N), rand(8, N)
    y = got.data[0].clone()
    for z in range(1, parts):
        y += got.data[z]
    h, r = ops.fused_add_rmsnorm(y.bfloat16(), res.clone(), norm, 1e-5)
    out, out_res = ops.fused_add_rmsnorm(got, res.clone(), norm, 1e-5)
    routed, routed_res = ops.fused_add_rmsnorm_route(got, res.clone(), norm, 1e-5,
                                                     router, 2)
    assert torch.equal(out_res, r) and torch.equal(routed_res, r)
    # the squares may be added in another order: the last bit of a row's scale
    for n in (out, routed.data):
        assert ((n.float() - h.float()).abs() <= h.float().abs() * 2.0 ** -7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(700, 16384, 1024), (1201, 6016, 3072),
                                   (1200, 14336, 3136)])
def test_gated_linear(M, N, K, monkeypatch):
    assert ops._wide_gated(M, N, K)
    x, w = _inputs(M, N, K)
    got = ops.gated_linear(x, w)
    monkeypatch.setattr(ops, "_wide_gated", lambda *a: None)
    want = ops.gated_linear(x, w).float()
    # one side rounds the halves to bf16 first
    assert (got.float() - want).norm() <= 2.0 ** -7 * want.norm()


@pytest.mark.gpu
def test_long_columns():
    M, N, K = 3600, 5120, 10240              # 300 tiles are 0.59 of two waves
    assert ops._wide_long(M, N, K) is None
    M = 5400                                 # 440 are 0.86
    high, bn, parts = ops._wide_long(M, N, K)
    assert parts == 1 and (high, bn) == (8, 256)
    x, w = _inputs(M, N, K)
    got, want = ops.linear(x, w).float(), x.float() @ w.float().t()
    assert (got - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.gpu
def test_refused():
    x, w = _inputs(300, 256, 128)
    out = torch.empty(300, 256, dtype=torch.bfloat16, device=DEV)
    part = torch.empty(2, 300, 256, device=DEV)
    wide = ops._native().gemm_wide
    for args in ((out, x, w, None, 3, 128), (out, x, w, None, 8, 64),
                 (None, x, w, None, 8, 128), (None, x, w, part, 8, 128, 3),
                 (None, x, w, part[:1], 8, 128, 2),
                 (out, x[:, :96], w[:, :96], None, 8, 128),
                 (out, x, w[:250], None, 8, 128),
                 (out[:, :128], x, w, None, 8, 128)):
        with pytest.raises(RuntimeError):
            wide(*args)


def test_rule_of_parts():
    """From 4608 columns on, up to 512 rows from 10240 on, in a nearly full wave;
    not in one part of tiles of 256 outputs."""
    for M, N, K, taken in [
            (600, 2048, 2048, False), (1024, 4096, 2560, False), (513, 2048, 4544, False),
            (600, 4096, 4608, True), (1025, 4096, 4608, False), (1024, 4096, 9216, True),
            (512, 4096, 9216, False), (512, 4096, 10240, True), (1400, 4096, 10240, True),
            (1401, 4096, 10240, False), (129, 4096, 14336, True),
            (128, 4096, 14336, False), (1114, 8144, 12928, False),
            (1028, 7992, 18624, False), (785, 6464, 18048, True)]:
        assert bool(ops._wide_parts(M, N, K)) == taken, (M, N, K)


def test_rule_of_gated_tiles():
    """The more rows, the shorter the columns."""
    for M, N, K, taken in [
            (257, 28672, 8192, True), (768, 28672, 8192, True),
            (769, 28672, 5440, False), (769, 28672, 5376, True),
            (1192, 16384, 5888, False), (901, 29712, 8064, False),
            (1200, 28672, 5376, True), (1201, 28672, 3136, False),
            (1201, 28672, 3072, True), (512, 28672, 4096, True),
            (512, 28672, 8256, False)]:
        assert bool(ops._wide_gated(M, N, K)) == taken, (M, N, K)


def test_rule_of_long_columns():
    """Two or three waves of 256 x 256 tiles, but not multiples of 64 of them."""
    for M, N, K, tiles, taken in [
            (6657, 4096, 11008, 27 * 16, True), (7041, 4096, 11008, 28 * 16, False),
            (7411, 4096, 14336, 29 * 16, True), (7680, 4096, 11008, 30 * 16, True),
            (7681, 4096, 11008, 31 * 16, False), (4353, 4096, 11008, 18 * 16, False),
            (6657, 6144, 16384, 27 * 24, True), (8960, 5120, 13824, 35 * 20, True),
            (8960, 4096, 13824, 35 * 16, False), (8193, 5120, 13824, 33 * 20, True),
            (7984, 7584, 18688, 32 * 30, False), (7489, 7256, 21120, 30 * 29, False),
            (16384, 2816, 14336, 64 * 11, False), (16380, 2560, 14336, 64 * 10, False),
            (16128, 2560, 14336, 63 * 10, True), (16385, 2560, 14336, 65 * 10, False)]:
        assert -(-M // 256) * -(-N // 256) == tiles
        assert bool(ops._wide_long(M, N, K)) == taken, (M, N, K)


def test_rules_cover_all_rows():
    """Every size that a rule takes has tiles that the kernel has, enough of them
    for all rows and outputs, and parts with columns."""
    rng = random.Random(1)
    taken = 0
    for _ in range(20000):
        M, N = rng.randint(1, 9000), rng.randint(1, 5000) * 8
        K = rng.randint(1, 400) * rng.choice([32, 64])
        for rule in (ops._wide_gated, ops._wide_parts, ops._wide_long):
            tile = rule(M, N, K)
            if tile is None:
                continue
            taken += 1
            high, bn, parts = (*tile, 1)[:3]
            assert M > (128 if rule is ops._wide_parts else 256)
            assert K % 64 == 0 and N % (
                16 if rule is ops._wide_gated else 8) == 0
            assert 4 <= high <= 8 and bn in (128, 256)
            assert 1 <= parts <= 8 and parts * 64 <= K
            assert parts == 1 or rule is ops._wide_parts
            # tiles are counted as they are launched, and are no more than needed
            every = range(1, 9) if rule is ops._wide_parts else (1,)
            counted = ops._wide_tile(M, N, K, tuple(every))
            assert counted[1:4] == (high, bn, parts)
            rows = -(-M // (32 * high))
            assert counted[4] == rows * -(-N // bn) * parts
            assert rows * 32 * high >= M > (rows - 1) * 32 * high
            assert rows <= -(-M // 256) + (M > 256)
            if parts > 1:
                assert counted[4] <= 256
    assert taken > 200
