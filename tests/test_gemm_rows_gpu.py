"""Products of few rows against float64 at the edges of tiles, batches and
what fits.

Bound: products of bf16 are exact in float; a sum of K of them is off by at
most K 2^-24 of the sum of magnitudes, and the result is rounded to bf16."""

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops
from hyperspot import _C

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("rows", [1, 3, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(16, 512), (20, 8), (260, 520), (4100, 1024),
                                 (8212, 264), (48, 4104), (36, 14336)])
def test_products_of_few_rows(rows, n, k):
    if not _C.gemm_rows_fits(rows, k):
        with pytest.raises(RuntimeError):
            _C.gemm_rows(torch.empty(rows, n, device=DEV).bfloat16(),
                         torch.empty(rows, k, device=DEV).bfloat16(),
                         torch.empty(n, k, device=DEV).bfloat16())
        return
    g = torch.Generator().manual_seed(rows * n)
    # rows of wider buffers
    x = torch.randn(rows, k + 8, generator=g).bfloat16().to(DEV)[:, :k]
    w = torch.randn(n, k + 16, generator=g).bfloat16() \
        .to(DEV)[:, 8:k + 8]
    out = torch.full((rows + 1, n + 4), 7.0, device=DEV).bfloat16()
    _C.gemm_rows(out[:rows, :n], x, w)
    assert (out[rows] == 7).all() and (out[:, n:] == 7).all()
    ref = x.double() @ w.double().t()
    slack = x.double().abs() @ w.double().abs().t() * k * 2.0 ** -24
    err = (out[:rows, :n].double() - ref).abs()
    assert (err <= slack + ref.abs() * 2.0 ** -8).all()


@pytest.mark.parametrize("rows", [0, 1, 64, 65])
def test_linear_takes_any_rows(rows):
    g = torch.Generator().manual_seed(5)
    x = torch.randn(rows, 1024, generator=g).bfloat16().to(DEV)
    w = torch.randn(2048, 1024, generator=g).bfloat16().to(DEV)
    ref = x.double() @ w.double().t()
    out = ops.linear(x, w).double()
    assert out.shape == ref.shape
    assert rows == 0 or (out - ref).norm() <= 2.0 ** -8 * ref.norm()


@pytest.mark.parametrize("rows", [1, 16, 20])
@pytest.mark.parametrize("n", [2044, 2052, 3068, 4096, 6144, 6148, 10244])
def test_heights_of_tiles(rows, n):
    """Tiles of 8, 12 and 16 rows of w, the last one whole or not."""
    test_products_of_few_rows(rows, n, 528)


@pytest.mark.parametrize("rows,k", [
    (1, 8), (1, 264), (1, 512), (1, 2056), (1, 4104), (16, 4104), (20, 8),
    (20, 264), (20, 1536), (20, 2056), (64, 1000)])
def test_infinities_in_the_last_columns(rows, k):
    """K is not a multiple of what a batch of loads covers."""
    g = torch.Generator().manual_seed(k)
    x = torch.randn(rows, k, generator=g).bfloat16()
    x[0, -1], x[-1, max(k - 9, 0)] = float("inf"), float("-inf")
    w = torch.randn(36, k, generator=g).bfloat16()
    w[w == 0] = 1
    ref = x.double() @ w.double().t()
    out = torch.empty(rows, 36, dtype=torch.bfloat16, device=DEV)
    _C.gemm_rows(out, x.to(DEV), w.to(DEV))
    out = out.double().cpu()
    odd = ~ref.isfinite()                      # NaN where both signs meet
    assert odd[0].all()
    assert torch.equal(out[odd].nan_to_num(0.0, 1.0, -1.0),
                       ref[odd].nan_to_num(0.0, 1.0, -1.0))
    assert out[~odd].isfinite().all()


def test_sizes_where_the_library_is_faster():
    """Rows of K that fill the loads in part, and outputs of a head or of a
    width that suits the library."""
    for m, n, k in ((16, 50304, 1024), (1, 50304, 512), (17, 6144, 2560),
                    (8, 7168, 3584), (16, 128256, 4096), (48, 16384, 512),
                    (8, 65536, 2304), (48, 4096, 1280), (4, 128256, 768)):
        assert not ops._rows_gemm_sizes(m, n, k)
    for m, n, k in ((16, 4096, 1024), (64, 4096, 768), (1, 4608, 2304),
                    (8, 32768, 4096), (32, 32768, 2048), (4, 7168, 4096),
                    (16, 28672, 3584), (48, 12288, 512), (16, 40960, 1536)):
        assert ops._rows_gemm_sizes(m, n, k)
