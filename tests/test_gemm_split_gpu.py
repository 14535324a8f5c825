"""Products of tens to hundreds of rows in parts of K, against float64.

Bound: the result is rounded to bf16 (2^-9 of it) and sums K products of float
precision in any order (K 2^-24 of the sum of their sizes)."""

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops

DEV = "cuda:0"


def _check(out, x, w):
    x, w = x.double().cpu(), w.double().cpu()
    ref = x @ w.t()
    bound = ref.abs() * 2.0 ** -8 \
        + x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().t())
    assert ((out.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", [(128, 64), (128, 128), (256, 128)])
@pytest.mark.parametrize("M,N,K,parts", [
    (1, 4, 128, 1), (31, 60, 256, 2), (128, 128, 384, 3), (129, 132, 640, 4),
    (256, 64, 1024, 8), (257, 260, 1152, 8), (97, 1028, 896, 7),
    (300, 516, 1408, 5), (33, 256, 2048, 6),
])
def test_gemm_split(M, N, K, parts, bm, bn):
    g = torch.Generator().manual_seed(M)
    # rows of both are views into wider ones
    x = torch.randn(M, K + 8, generator=g).bfloat16().to(DEV)[:, :K]
    w = torch.randn(N, K + 16, generator=g).bfloat16().to(DEV)[:, 16:]
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    part = torch.full((parts * M * N,), float("nan"), device=DEV)
    ops._native().gemm_split(out, x, w, part, bm, bn, parts)
    _check(out, x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", [(64, 64), (64, 128)])
@pytest.mark.parametrize("M,N,K,parts", [
    (1, 4, 128, 1), (64, 60, 256, 2), (65, 132, 640, 4), (33, 1028, 896, 7)])
def test_tiles_of_64_rows(M, N, K, parts, bm, bn):
    test_gemm_split(M, N, K, parts, bm, bn)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 2048, 7168), (16, 4096, 14336),
                                   (1, 416, 5120), (16, 3264, 5120),
                                   (9, 5440, 8704), (7, 3272, 6784),
                                   (33, 2048, 2048), (64, 4096, 1280),
                                   (128, 4096, 2560), (257, 3200, 8192),
                                   (480, 4096, 4096), (400, 5120, 5120)])
def test_parts_that_the_norm_adds_up(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    bm, bn, parts = ops._summed_gemm(M, N, K)
    assert -(-M // bm) * -(-N // bn) * parts <= 256 and 1 < parts <= 8
    got = ops.linear_parts(x, w)
    assert got.data.shape == (parts, M, N)
    _check(got.data.sum(0), x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 63, 64, 65])
@pytest.mark.parametrize("N,K", [(11204, 128), (16384, 384), (16388, 256),
                                 (22404, 640), (32768, 256), (32772, 128)])
def test_one_wave_of_tiles(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    assert (ops._wave_gemm(M, N, K) is None) == (
        M > 64 or N in (16388, 32772))
    _check(ops.linear(x, w), x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 128), (31, 120, 256), (64, 128, 384), (65, 264, 640), (128, 1032, 128),
    (129, 8, 1024), (17, 4104, 512)])
def test_gated(M, N, K, bm, bn):
    """silu(gate) * up: an error e of the gate becomes at most 1.1 e |up|, one of
    up |silu| e; the result is rounded to bf16 and the exponential is exact to
    2^-20."""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K + 8, generator=g).bfloat16().to(DEV)[:, :K]
    w = (torch.randn(N, K, generator=g) * 0.1).bfloat16().to(DEV)
    out = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16,
                     device=DEV)
    ops._native().gemm_split(out, x, w, None, bm, bn, 1, gated=True)
    x, w = x.double().cpu(), w.double().cpu()
    gate, up = (x @ w.t()).chunk(2, -1)
    err = K * 2.0 ** -24 * (x.abs() @ w.abs().t())
    silu = torch.nn.functional.silu(gate)
    ref = silu * up
    bound = ref.abs() * 2.0 ** -8 + 1.1 * up.abs() * err[:, :N // 2] \
        + silu.abs() * err[:, N // 2:] + 1e-30
    assert ((out.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 64, 65, 128, 129, 256, 257])
@pytest.mark.parametrize("N,K", [(2048, 1024), (14336, 2048), (28672, 512),
                                 (28672, 4224), (2064, 640)])
def test_gated_linear(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    out = ops.gated_linear(x, w)
    want = ops.silu_mul(x @ w.t())      # gate and up rounded to bf16
    tile = ops._gated_tile(M, N, K)
    assert tile is None or M <= 256
    assert (out.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (1, 16, 128), (129, 136, 256), (256, 1040, 384), (257, 240, 512),
    (512, 264, 640), (300, 4112, 128)])
def test_gated_in_tiles_of_256_rows(M, N, K):
    """One to five stages of the ring; the bound as in test_gated."""
    test_gated(M, N, K, 256, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (129, 16528, 256), (256, 32768, 640), (257, 16384, 128), (512, 6144, 1024)])
def test_gated_wave(M, N, K):
    assert ops._gated_tile(M, N, K) is None
    assert ops._gated_wave(M, N, K) == (256, 128)
    assert ops._gated_wave(M, 32768 + 16, 4608) is None
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    out, want = ops.gated_linear(x, w), ops.silu_mul(x @ w.t())
    assert (out.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,tiles", [
    ("bf16", [(64, 64), (64, 128), (128, 64)]),
    ("gated", [(64, 64), (64, 128), (128, 64), (128, 128)]),
    ("e4m3", [(64, 32), (64, 64), (64, 128)])])
def test_equal_rows_have_equal_bits(kind, tiles):
    """In whatever tile of rows they are, whose workgroups begin at the same
    column."""
    M, N, K = 300, 2064, 1280
    g = torch.Generator().manual_seed(3)
    x = torch.randn(1, K, generator=g).bfloat16().expand(M, K).contiguous() \
        .to(DEV)
    w = (torch.randn(N, K, generator=g) * 0.1).bfloat16().to(DEV)
    scales = ()
    if kind == "e4m3":
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        scales = (torch.ones(M, device=DEV), torch.ones(N, device=DEV))
    for bm, bn in tiles:
        out = torch.empty(M, N // 2 if kind == "gated" else N,
                          dtype=torch.bfloat16, device=DEV)
        ops._native().gemm_split(out, x, w, None, bm, bn, 1, *scales,
                                 gated=kind == "gated")
        assert torch.equal(out, out[:1].expand_as(out)), (bm, bn)


@pytest.mark.gpu
def test_gated_linear_rows_far_apart():
    """Up rows that 32 bits of offset do not reach from the gate rows."""
    M, N, K, far = 17, 2560, 256, 1 << 21
    assert ops._gated_tile(M, N, K) is not None
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = torch.empty(N * far, device=DEV, dtype=torch.bfloat16).view(N, far)[:, :K]
    w.normal_(0, K ** -0.5)
    assert torch.equal(ops.gated_linear(x, w), ops.silu_mul(ops.linear(x, w)))


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [1 << 22, (1 << 22) + 8])
def test_rows_far_apart(stride, monkeypatch):
    """Up to where 32 bits of offset reach the last row of a tile; one row of x,
    whose stride means nothing."""
    M, N, K = 17, 132, 640
    x = torch.empty(M * stride, device=DEV, dtype=torch.bfloat16).view(
        M, stride)[:, :K].normal_()
    w = torch.randn(N, K, device=DEV).bfloat16()
    monkeypatch.setattr(ops, "_route", lambda *a: (64, 64, 2))
    seen = []
    kernel = ops._native().gemm_split
    monkeypatch.setattr(ops._native(), "gemm_split", lambda *a: (
        seen.append(1), kernel(*a)))
    _check(ops.linear(x, w), x, w)
    one = x[:1].as_strided((1, K), (1 << 40, 1))
    _check(ops.linear(one, w), one, w)
    assert len(seen) == 2


def test_reach_of_a_tile():
    """The farthest rows that 32 bits of offset reach, and the next ones."""
    for dtype, size in ((torch.bfloat16, 2), (torch.float8_e4m3fn, 1)):
        near = torch.empty(8, 128, dtype=dtype, device="meta")
        for rows in (1, 2, 64, 65, 300):
            for stride in (1 << 22, 1 << 25, 1 << 26, 1 << 40):
                far = torch.empty_strided((rows, 128), (stride, 1),
                                          dtype=dtype, device="meta")
                last = (min(rows, 64) - 1) * stride * size + 256
                assert ops._near(far, near, 64, 128) == (last < 1 << 32)
                assert ops._near(near, far, 128, 64) == (last < 1 << 32)


@pytest.mark.gpu
def test_watched_products_get_their_calls():
    """A hook on the gate and up product sees it, and may change it."""
    from hyperspot.engine.config import ModelSpec
    from hyperspot.models.llama import LlamaMLP
    from hyperspot.parallel import layers
    layers.set_init_device(DEV)
    spec = ModelSpec("t", 256, 1, 2, 1, 128, 2048, 32)
    mlp = LlamaMLP(spec, 0, torch.bfloat16).to(DEV)
    layers.set_init_device("cpu")
    x = torch.randn(32, 256, device=DEV).bfloat16()
    fused = mlp(x)
    seen = []
    h = mlp.gate_up.register_forward_hook(
        lambda m, a, y: seen.append(y.shape) or y * 0)
    assert mlp(x).abs().max() == 0 and seen == [(32, 4096)]
    h.remove()
    assert torch.equal(mlp(x), fused)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 128, 129, 256, 257, 512])
@pytest.mark.parametrize("N,K", [(4096, 4096), (2048, 7168), (5120, 8192)])
def test_linear_takes_it(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    out = ops.linear(x, w)
    _check(out, x, w)
    route = "rows" if M == 17 and K == 4096 \
        else "library" if M > 256 and (N, K) != (2048, 7168) else "split"
    rule = ops._route(M, N, K, False)
    assert (rule == "rows") == (route == "rows")
    assert (rule is None) == (route == "library")
    if (M, N, K) == (17, 2048, 7168):
        assert rule[:2] == (64, 64)
    again = torch.empty_like(out)
    if route == "rows":
        ops._native().gemm_rows(again, x, w)
    elif route == "library":
        again = x @ w.t()
    else:
        part = torch.empty(rule[2] * M * N, device=DEV)
        ops._native().gemm_split(again, x, w, part, *rule)
    assert torch.equal(out, again)


@pytest.mark.gpu
def test_one_wave_goes_before_rows():
    """Where both rules would take a product of few rows."""
    M, N, K = 4, 16384, 2048
    assert ops._rows_gemm_sizes(M, N, K) and ops._native().gemm_rows_fits(M, K)
    assert ops._route(M, N, K, False) == ops._wave_gemm(M, N, K) == (64, 64, 1)
    x, w = (torch.randn(n, K, device=DEV).bfloat16() for n in (M, N))
    again = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops._native().gemm_split(again, x, w, None, 64, 64, 1)
    assert torch.equal(ops.linear(x, w), again)


def test_rule_stays_in_what_the_kernel_takes():
    taken = 0
    for M in range(1, 600, 5):
        for N in (4, 512, 1000, 2048, 3072, 4096, 6144, 8192, 28672, 1 << 17):
            for K in (128, 4096, 4160, 7168, 8192, 14336, 1 << 16):
                rule = ops._split_gemm(M, N, K)
                if rule is None:
                    continue
                taken += 1
                bm, bn, parts = rule
                assert (bm, bn) in ((128, 64), (128, 128), (256, 128))
                assert 1 <= parts <= min(8, K // 128) and K % 128 == 0
                assert -(-M // bm) * -(-N // bn) * parts <= 256
    assert taken


def test_rule_of_few_rows_of_long_columns():
    """From 5 parts on, or with 3 where the library has no better tile; as
    many workgroups as units at most."""
    taken = lambda N, K: ops._summed_gemm(8, N, K) is not None
    assert taken(3264, 5120) and not taken(3272, 5120) and not taken(3264, 4992)
    assert taken(3272, 6784) and not taken(3272, 7168) and taken(3272, 9216)
    assert taken(2048, 16384) and not taken(4096, 16384)
    assert not taken(5504, 9216)
    for N in range(8, 8193, 104):
        for K in range(5120, 20481, 128):
            rule = ops._summed_gemm(8, N, K)
            if rule is not None:
                assert -(-N // 64) * rule[2] <= 256 and 3 <= rule[2] <= K // 512


def test_rule_of_few_parts_of_one_tile():
    """Up to 64 rows: at most a workgroup a unit; what rows of 16 KB took is right for
    them by now, and few parts of many columns are not narrow ones."""
    few2, few3, four, wide = (64, 64, 2), (64, 64, 3), (64, 64, 4), (128, 128, 8)
    for M, N, K, few, narrow in [
            (1, 8192, 28672, few2, None), (64, 8192, 4224, few2, None),
            (64, 8192, 4096, None, None), (1, 8192, 8192, few2, None),
            (1, 8192, 28800, None, None), (65, 8192, 28672, None, None),
            (8, 5440, 8192, few3, None), (8, 5448, 9216, few2, None),
            (8, 4096, 9216, None, None), (8, 8196, 9216, None, None),
            (1, 5120, 5120, few3, None), (1, 4992, 5120, None, None),
            (2, 4608, 4608, None, None), (2, 4608, 4736, few3, None),
            (1, 4168, 5376, few3, None), (33, 4096, 11008, None, four),
            (33, 4096, 8192, None, four), (48, 4096, 18432, None, four),
            (48, 4096, 18560, None, wide), (49, 4096, 12288, None, four),
            (49, 4096, 14336, None, wide), (17, 1088, 16384, None, (64, 64, 8)),
            (64, 5120, 8192, few3, few3), (64, 5120, 12288, few3, (128, 128, 6)),
            (48, 5120, 12288, few3, few3), (48, 5120, 12416, few3, (128, 128, 6)),
            (17, 6144, 6144, few2, (128, 128, 5))]:
        assert ops._few_parts(M, N, K) == few, (M, N, K)
        assert ops._less_padding(M, N, K, ops._split_gemm(M, N, K)) == narrow
        route = ops._route(M, N, K, True)
        assert route == (narrow or few or route), (M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (1, 8192, 4224), (64, 6592, 9216), (7, 4168, 4480), (33, 4096, 11008),
    (17, 1088, 16384), (64, 5120, 6272), (40, 3080, 8192)])
def test_parts_of_one_tile_of_rows(M, N, K):
    """Workgroups of a tile of w begin at a column of its own in each part."""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    bm, bn, parts = ops._route(M, N, K, True)
    assert bm == bn == 64 and -(-N // 64) * parts <= 256
    got = ops.linear_parts(x, w)
    assert got.data.shape == (parts, M, N)
    _check(got.data.sum(0), x, w)
    # where it begins depends on how far the rows of w lie apart, but for 32 KB more
    pad = lambda t, n: torch.nn.functional.pad(t, (0, n))[:, :K]
    assert torch.equal(ops.linear_parts(pad(x, 8), pad(w, 16384)).data, got.data)
    _check(ops.linear_parts(pad(x, 8), pad(w, 8)).data.sum(0), x, w)
    # a row alone, where it has as many parts, has the same sums
    alone = {1088: 6}.get(N, parts)
    assert ops._route(1, N, K, True) == (64, 64, alone)
    one = ops.linear_parts(x[M - 1:], w)
    assert one.data.shape == (alone, 1, N)
    if alone == parts:
        assert torch.equal(one.data[:, 0], got.data[:, M - 1])
    else:
        _check(one.data.sum(0), x[M - 1:], w)


def test_rule_of_several_waves():
    """Half a wave and more, and several; not nearly empty ones."""
    for M, N, K, rule in [
            (1, 9152, 2048, None), (1, 9153 + 3, 2048, "rows"),
            (5, 9156, 2048, (64, 64, 1)), (1, 9156, 1024, (64, 64, 1)),
            (4, 9156, 5120, "rows"), (4, 9156, 5248, (64, 64, 1)),
            (64, 11264, 640, None), (64, 11200, 512, None),
            (5, 16388, 2048, (64, 128, 1)), (64, 22400, 768, (64, 128, 1)),
            (1, 33000, 2048, None), (1, 45000, 1024, None),
            (5, 45000, 1152, (64, 64, 1)), (17, 45000, 1152, None),
            (16, 49156, 896, (64, 128, 1)), (1, 49156, 768, None),
            (32, 65700, 640, (64, 128, 1)), (5, 69632, 2048, (64, 64, 1)),
            (32, 49156, 1024, None), (64, 128256, 4096, (64, 128, 1)),
            (64, 128256, 4224, None), (64, 69632, 1024, None),
            (65, 128256, 4096, None), (1, 128256, 4100, None)]:
        assert ops._waves_gemm(M, N, K) == rule, (M, N, K)


def test_rules_leave_what_no_tile_takes():
    """Tiles count up to 2^24 outputs, the kernel of few rows up to 2^31."""
    for M in (1, 4, 5, 8, 16, 17, 32, 33, 64, 65, 192, 256, 512):
        for N in (1 << 24, (1 << 24) + 128, 3 << 23, 1 << 25):
            for K in (128, 640, 1024, 1152, 2048, 4096, 5120, 16384):
                for parts in (False, True):
                    assert ops._route(M, N, K, parts) in (None, "rows")
                assert ops._gated_tile(M, N, K) is None
                assert ops._gated_wave(M, N, K) is None
    # a product that the tiles still take, and the first that they do not
    assert ops._route(8, (1 << 24) - 4, 1152, False) == (64, 128, 1)
    assert ops._route(8, 1 << 24, 1152, False) == \
        ("rows" if ops._rows_gemm_sizes(8, 1 << 24, 1152) else None)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (1, 9156, 640), (64, 11196, 896), (33, 16388, 640), (16, 22396, 768),
    (3, 45000, 1152), (17, 65668, 640), (64, 75268, 640), (5, 69644, 896)])
def test_several_waves(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    assert ops._route(M, N, K, False) == ops._waves_gemm(M, N, K) is not None
    _check(ops.linear(x, w), x, w)


def test_rule_of_one_tile_of_rows():
    """129 to 256 rows: one tile of 256 from as many columns on as pay for the
    parts, which fill the units; not where narrower ones have five parts."""
    for M, N, K, rule in [
            (256, 4096, 14336, (128, 128, 4)), (129, 4096, 15360, (256, 128, 8)),
            (129, 4104, 8832, (128, 128, 3)), (256, 3200, 16384, (128, 128, 5)),
            (200, 4104, 8960, (256, 128, 7)), (200, 8192, 4608, (256, 128, 4)),
            (200, 8192, 4480, (128, 64, 1)), (200, 10880, 4096, (256, 128, 3)),
            (200, 10888, 6656, None), (200, 16384, 6784, (256, 128, 2)),
            (200, 16388, 6784, None), (257, 16384, 8192, None)]:
        assert ops._split_gemm(M, N, K) == rule, (M, N, K)
    assert ops._summed_gemm(512, 6504, 8704) == (256, 128, 2)
    assert ops._summed_gemm(512, 6504, 8576) is None


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(129, 4096, 15360), (256, 16384, 6784),
                                   (255, 4104, 9088), (200, 8196, 4096),
                                   (145, 8188, 4608)])
def test_one_tile_of_rows(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    assert ops._route(M, N, K, False)[:2] == (256, 128)
    _check(ops.linear(x, w), x, w)


def test_rule_of_a_wave_of_rows():
    """65 to 192 rows: 144 to 256 tiles, none for a second wave on any die."""
    for M, N, K, rule in [
            (65, 4608, 384, (64, 64, 1)), (65, 4544, 2048, None),
            (128, 8192, 2304, (64, 64, 1)), (128, 8196, 2048, None),
            (128, 8192, 2432, None), (192, 3072, 2048, (64, 64, 1)),
            (129, 5120, 640, (64, 64, 1)), (129, 5124, 640, None),
            (193, 3072, 2048, None), (64, 8192, 640, None),
            (128, 8192, 256, None), (128, 8192, 700, None),
            (128, 8190, 640, None)]:
        assert ops._wave_of_rows(M, N, K) == rule, (M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (65, 4612, 384), (128, 8188, 640), (129, 3204, 2304), (192, 5120, 896)])
def test_wave_of_rows(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    assert ops._route(M, N, K, False) == ops._wave_of_rows(M, N, K) is not None
    _check(ops.linear(x, w), x, w)


def test_rule_of_a_wave_of_longer_rows():
    """65 to 128 rows: 176 to 256 tiles, without a norm that adds up parts and where
    there are none of 128 x 128 either."""
    for M, N, K, rule in [
            (65, 5632, 2432, (64, 64, 1)), (65, 5568, 4096, None),
            (128, 8192, 4608, (64, 64, 1)), (128, 8196, 4096, None),
            (96, 6144, 4736, None), (96, 6144, 2304, None),
            (97, 6144, 3712, None), (125, 6032, 2560, None),
            (97, 6144, 3840, (64, 64, 1)), (128, 6144, 5120, None),
            (129, 6144, 4096, None), (64, 6144, 4096, None),
            (96, 6144, 4160, None), (96, 6142, 4096, None)]:
        assert ops._wave_of_longer_rows(M, N, K) == rule, (M, N, K)
    for M, N, K in [(66, 6144, 4096), (96, 6144, 4096), (128, 6528, 4608)]:
        for parts in (True, False):
            assert ops._route(M, N, K, parts) == ops._split_gemm(M, N, K) \
                == (128, 128, 5)
    for M, N, K in [(66, 6656, 4096), (128, 6144, 3968), (96, 8192, 4608)]:
        assert ops._route(M, N, K, False) == (64, 64, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 5572, 2432), (96, 6656, 4096),
                                   (128, 8188, 4608)])
def test_wave_of_longer_rows(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    assert ops._route(M, N, K, False) == (64, 64, 1)
    _check(ops.linear(x, w), x, w)
    apart = [torch.nn.functional.pad(t, (0, 8))[:, :K] for t in (x, w)]
    assert torch.equal(ops.linear(*apart), ops.linear(x, w))


def test_rule_leaves_no_workgroup_for_a_second_wave():
    """Workgroups go to 8 dies of 32 units in turn, those of one tile of w to
    the same."""
    for M in range(17, 513, 5):
        for N in range(512, 9000, 132):
            for K in (4096, 7168, 8192, 13824):
                rule = ops._split_gemm(M, N, K)
                if rule is None:
                    continue
                bm, bn, parts = rule
                assert -(-(-(-N // bn) * parts) // 8) * -(-M // bm) <= 32
    assert ops._split_gemm(384, 2688, 7552) == (256, 128, 6)


def test_sizes_where_the_library_is_faster():
    for m, n, k in ((257, 3072, 8192), (17, 4096, 16384), (17, 1024, 8192),
                    (144, 7168, 7168)):
        assert ops._split_gemm(m, n, k) is None
    for m, n, k in ((321, 3072, 8192), (257, 3584, 8192), (64, 4096, 16384),
                    (144, 6144, 7168), (145, 7168, 7168)):
        assert ops._split_gemm(m, n, k) is not None


def test_rules_leave_sizes_beyond_the_kernel_to_the_library(monkeypatch):
    """No columns, and sizes from 2^24 on."""
    monkeypatch.setattr(ops, "_native", lambda: type("", (), {
        "gemm_rows_fits": staticmethod(lambda M, K: True)}))
    ops._route.cache_clear()
    for M in (0, 1, 16, 17, 64, 65, 128, 256, 512):
        for N, K in ((16384, 0), (28672, 0), (4096, 0), (0, 4096), (0, 0),
                     (8, 1 << 24), (4096, 1 << 24), (1 << 24, 128)):
            for parts in (False, True):
                route = ops._route(M, N, K, parts)
                assert route is None or route == "rows" and N * K, (M, N, K)
                assert ops._tiles_q(M, N, K, parts) is None
            assert ops._gated_tile(M, N, K) is None, (M, N, K)
    ops._route.cache_clear()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(1, 16384), (17, 28672), (64, 4096)])
def test_products_of_no_columns(M, N):
    x, w = (torch.empty(n, 0, dtype=torch.bfloat16, device=DEV) for n in (M, N))
    assert torch.equal(ops.linear(x, w), x @ w.t())
    assert torch.equal(ops.linear_parts(x, w), x @ w.t())
    assert torch.equal(ops.gated_linear(x, w), ops.silu_mul(x @ w.t()))


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,pad,parts,fp8,apart", [
    (4096, 14336, 0, 4, False, False), (4096, 14336, 2048, 4, False, True),
    (4096, 14336, 0, 4, True, False), (5120, 8192, 0, 3, False, True),
    (5120, 8192, 64, 3, False, False), (5120, 6144, 0, 3, False, True),
    (5120, 6144, 64, 3, False, False), (5120, 12288, 0, 3, True, True),
    (2560, 9472, 0, 6, True, False), (8192, 12288, 0, 2, False, True),
    (8192, 14336, 0, 2, False, False), (4096, 12288, 0, 4, False, False)])
def test_where_parts_begin(N, K, pad, parts, fp8, apart):
    """Tiles of w begin at columns of their own where rows and parts would begin on few
    channels of memory, by what lies between rows; elsewhere at the same, so that their
    sums do not depend on where among the outputs they are."""
    g = torch.Generator().manual_seed(K)
    x = torch.randn(5, K, generator=g)
    w = torch.randn(N, K + pad, generator=g)
    scales = ()
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        scales = torch.ones(5, device=DEV), torch.ones(N, device=DEV)
    else:
        x, w = x.bfloat16(), w.bfloat16()
    x, w = x.to(DEV), w.to(DEV)

    def product(w):
        part = torch.full((parts, 5, N), float("nan"), device=DEV)
        ops._native().gemm_split(None, x, w[:, :K], part, 64, 64, parts, *scales)
        return part

    got = product(w)
    other = product(w.view(torch.uint8).roll(64, 0).view(w.dtype))
    same = torch.equal(other.roll(-64, 2), got)
    assert same or apart
    if not fp8:                 # whose sums are exact here in any order
        assert same != apart
        _check(got.sum(0), x, w[:, :K])
    ref = x.double() @ w[:, :K].double().t()
    assert (got.sum(0).double() - ref).norm() <= 2.0 ** -14 * ref.norm()
