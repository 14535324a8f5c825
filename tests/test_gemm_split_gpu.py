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
@pytest.mark.parametrize("M", [17, 128, 129, 256, 257, 512])
@pytest.mark.parametrize("N,K", [(4096, 4096), (2048, 7168), (5120, 8192)])
def test_linear_takes_it(M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    _check(ops.linear(x, w), x, w)


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
