"""Op dispatch layer.

On GPU (ROCm) every hot op runs a hand-written CDNA4 HIP kernel from the
in-tree extension ``hyperspot._C`` (csrc/, built for gfx950 only).  On CPU the
pure-PyTorch references in :mod:`hyperspot.ops.torch_ref` run instead (CI has
no GPU).  There is no CUDA path, no Triton, no multi-backend dispatch — a CUDA
device without the extension is a hard error, never a silent eager fallback.
"""

from __future__ import annotations

from functools import lru_cache
from typing import NamedTuple, Optional

import torch

from . import torch_ref

_C = None
_C_ERR: Exception | None = None
try:  # built by `python csrc/setup.py build_ext --inplace` (gfx950)
    from hyperspot import _C as _C  # type: ignore
except Exception as e:  # pragma: no cover - exercised only on GPU boxes
    _C_ERR = e


def have_native() -> bool:
    return _C is not None


def _native():
    if _C is None:
        raise RuntimeError(
            "hyperspot._C (gfx950 HIP extension) is not built but a GPU tensor "
            "reached the op layer. Build it in-tree with "
            "`python csrc/setup.py build_ext --inplace` "
            f"(import error: {_C_ERR!r})")
    return _C


class Parts(NamedTuple):
    """A product whose sum over parts of K is still to be formed: data
    [parts, rows, outputs] float."""

    data: torch.Tensor


class Choices(NamedTuple):
    """Outputs of experts whose weighted sum is still to be formed: row t is the
    sum over k of weights[t, k] * data[place[t, k]], without those of place
    -1."""

    data: torch.Tensor
    place: torch.Tensor          # [T, K] int32
    weights: torch.Tensor        # [T, K] float


class Routed(NamedTuple):
    """Rows with the experts that they choose."""

    data: torch.Tensor           # [T, W]
    weights: torch.Tensor        # [T, K] float
    ids: torch.Tensor            # [T, K] int32


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().rmsnorm(out, x, weight, eps)
        return out
    return torch_ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor,
                      weight: torch.Tensor, eps: float):
    """residual += x (in place); x_out = rmsnorm(residual) (in place on x).

    x may be the Parts of a product or the Choices of experts, which are added
    up on the way."""
    if isinstance(x, Choices):
        out = torch.empty_like(residual)
        _native().choices_add_rmsnorm(out, x.data, x.place, x.weights,
                                      residual, weight, eps)
        return out, residual
    if isinstance(x, Parts):
        out = torch.empty_like(residual)
        _native().parts_add_rmsnorm(out, x.data, residual, weight, eps)
        return out, residual
    if x.is_cuda:
        _native().fused_add_rmsnorm(x, residual, weight, eps)
        return x, residual
    out, res = torch_ref.fused_add_rmsnorm(x, residual, weight, eps)
    return out, res


def fused_add_rmsnorm_route(x, residual: torch.Tensor, weight: torch.Tensor,
                            eps: float, router: torch.Tensor, top: int,
                            slots: Optional[torch.Tensor] = None):
    """fused_add_rmsnorm, x a tensor or Parts, and moe_router in one kernel:
    (Routed, residual); residual is changed in place.  Rows of a negative slot
    (int64) choose no expert.  GPU."""
    data = x.data if isinstance(x, Parts) else x
    T, W = residual.shape
    out = torch.empty_like(residual)
    share = torch.empty(T, top, dtype=torch.float32, device=residual.device)
    ids = torch.empty(T, top, dtype=torch.int32, device=residual.device)
    _native().norm_router(share, ids, out, data, residual, weight, eps, router,
                          top, slots)
    return Routed(out, share, ids), residual


def rope_kv_append(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                   positions: torch.Tensor, cos_sin: torch.Tensor,
                   slot_mapping: torch.Tensor,
                   k_cache: torch.Tensor, v_cache: torch.Tensor) -> None:
    """Fused: NeoX RoPE on q,k (in place) + scatter k,v into the paged cache.

    q [T,H,D], k/v [T,KV,D]; cos_sin [max_pos, D] fp32 (cos half | sin half);
    slot_mapping [T] int64 (-1 = skip append, e.g. sliding-window drop).
    """
    if q.is_cuda:
        _native().rope_kv_append(q, k, v, positions, cos_sin, slot_mapping,
                                 k_cache, v_cache)
        return
    d = q.shape[-1]
    cs = cos_sin[positions.long()]
    cos, sin = cs[:, : d // 2], cs[:, d // 2:]
    q.copy_(torch_ref._rotate_neox(q, cos, sin))
    k.copy_(torch_ref._rotate_neox(k, cos, sin))
    mask = slot_mapping >= 0
    if mask.any():
        torch_ref.kv_cache_append(k[mask], v[mask], k_cache, v_cache,
                                  slot_mapping[mask])


import os

_ATTN_SPLIT_TARGET = int(os.environ.get("HYPERSPOT_ATTN_SPLIT_TARGET", "256"))


def _attn_split(rows: int, kvh: int) -> int:
    """Flash-decode page-split factor: bring the workgroup count up to
    ~_ATTN_SPLIT_TARGET when rows*kvh alone cannot fill the 256 CUs (small
    batch, or the kvh=1 GQA shard of 70B at TP=8).  At 256 workgroups and
    more the partial round trip and the merge cost more than they buy.  us for
    1, 2, 4, 8, 16 parts: 1 row x 8 kv heads of 8000 tokens 89 51 31 21 18;
    8 x 8 of 8000 130 79 61 62 65; 32 x 4 of 1000 25 23 24 26 29; 64 x 8 of
    1000 59 64 66.  Static in (rows, kvh) => capture-safe."""
    s = max(1, min(16, _ATTN_SPLIT_TARGET // max(1, rows * kvh)))
    return 1 if s <= 1 else s


def _attn_parts(q: torch.Tensor, kvh: int) -> tuple:
    """(workspace or None, parts) of decode attention."""
    split = _attn_split(q.shape[0], kvh) if q.shape[-1] == 128 else 1
    if split == 1:
        return None, 1
    return torch.empty(q.shape[0] * split * q.shape[1] * 130,
                       dtype=torch.float32, device=q.device), split


def paged_attn_decode(q: torch.Tensor, k_cache: torch.Tensor,
                      v_cache: torch.Tensor, block_tables: torch.Tensor,
                      seq_lens: torch.Tensor, scale: float) -> torch.Tensor:
    if q.is_cuda:
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        ws, split = _attn_parts(q, k_cache.shape[1])
        _native().paged_attn(out, q, k_cache, v_cache, block_tables,
                             seq_lens, None, scale, ws, split)
        return out
    return torch_ref.paged_attn_decode(q, k_cache, v_cache, block_tables,
                                       seq_lens, scale)


# Portions of at least this many rows attend on tiles of 32 rows, the others row
# by row.  A tile takes a context's latency whatever it holds, a row its share
# of the memory: one portion of 16, 64, 96, 112 rows after 1000 tokens takes 36,
# 39, 41, 41 us in tiles and 16, 28, 38, 47 by rows, after 16000 491, 494, 495,
# 494 and 144, 284, 418, 555 (8 kv heads of 4; with e4m3 pages 112 and 192 rows
# after 1000 44, 46 and 34, 49).  Beside others tiles share the latency: 8
# portions of 4, 8, 16 rows 41, 37, 37 us and 25, 44, 48.
PORTION_ROWS, PORTION_ROWS_ALONE = 16, 104


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
              k_cache: torch.Tensor, v_cache: torch.Tensor, meta,
              scale: float) -> torch.Tensor:
    """Attention for one layer, prefill or decode.

    Decode rows attend over their seq_len cache slots.  Whole prompts attend
    over k and v as they came from the projection; portions whose earlier
    tokens are cached attend over slots 0..pos of the pages (their own k/v
    were appended by the fused RoPE kernel just before).
    """
    if meta.mode == "decode":
        return paged_attn_decode(q, k_cache, v_cache, meta.block_tables,
                                 meta.seq_lens, scale)
    if q.is_cuda:
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        if q.shape[-1] == 128 and getattr(meta, "fresh_prefill", True):
            # MFMA flash prefill (K/V straight from the qkv projection)
            _native().attn_prefill_mfma(out, q, k, v, meta.seq_start,
                                        meta.max_seqlen, scale)
        elif q.shape[-1] == 128 and meta.seq_start is not None \
                and q.shape[1] // k_cache.shape[1] in (1, 2, 4, 8) \
                and k_cache.data_ptr() % 16 == v_cache.data_ptr() % 16 == 0:
            least = PORTION_ROWS_ALONE if q.shape[0] < PORTION_ROWS_ALONE \
                else PORTION_ROWS
            _native().attn_portions(
                out, q, k_cache, v_cache, meta.block_tables, meta.ctx_lens,
                meta.row_seq, meta.seq_start, least,
                getattr(meta, "min_seqlen", 0) < least, scale)
        else:
            # row by row: odd head dims, pages that begin off 16 bytes
            _native().paged_attn(out, q, k_cache, v_cache,
                                 meta.block_tables, meta.ctx_lens,
                                 meta.row_seq, scale, None, 1)
        return out
    if getattr(meta, "fresh_prefill", True):
        return torch_ref.prefill_attn(q, k, v, meta.seq_start, scale)
    return torch_ref.prefill_attn_paged(q, k_cache, v_cache,
                                        meta.block_tables, meta.ctx_lens,
                                        meta.row_seq, scale)


def _rope_in_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                       k_cache: torch.Tensor, meta) -> bool:
    """Whether one launch turns, appends and attends: decoded tokens, heads as
    the matrix-core kernel takes them, rows that it can read 16 bytes at a
    time.  It is faster than two for one row of 1000 tokens (10.1 and 12.6 us)
    as for 256 rows of 30 (21.9 and 22.4) or 1000 (206 and 221)."""
    return q.is_cuda and meta.mode == "decode" and q.shape[-1] == 128 \
        and k_cache.shape[2] == 16 \
        and q.shape[1] // k.shape[1] in (1, 2, 3, 4, 8) \
        and all(t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0
                for t in (q, k, v))


def rope_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                   positions: torch.Tensor, cos_sin: torch.Tensor,
                   slot_mapping: torch.Tensor, k_cache: torch.Tensor,
                   v_cache: torch.Tensor, meta, scale: float) -> torch.Tensor:
    """rope_kv_append, then attention; q and k may be left turned or not."""
    if _rope_in_attention(q, k, v, k_cache, meta):
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        ws, split = _attn_parts(q, k.shape[1])
        _native().rope_paged_attn(out, q, k, v, positions, cos_sin,
                                  slot_mapping, k_cache, v_cache,
                                  meta.block_tables, meta.seq_lens, scale,
                                  ws, split)
        return out
    rope_kv_append(q, k, v, positions, cos_sin, slot_mapping, k_cache,
                   v_cache)
    return attention(q, k, v, k_cache, v_cache, meta, scale)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    if gate_up.is_cuda:
        i = gate_up.shape[-1] // 2
        out = torch.empty(*gate_up.shape[:-1], i, dtype=gate_up.dtype,
                          device=gate_up.device)
        _native().silu_mul(out, gate_up)
        return out
    return torch_ref.silu_mul(gate_up)


def unrecorded(*tensors: torch.Tensor) -> bool:
    """Whether a kernel may take the place of torch's operation on these: no
    gradient or tangent is formed, and no subclass, transform, trace or mode
    has to see the operation."""
    if torch.compiler.is_compiling() or _forward_ad._current_level >= 0 \
            or _stack() is not None or _modes() or _tracing() is not None \
            or torch.is_autocast_enabled("cuda"):
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:       # a loop: every product of a step comes here
        if type(t) not in _PLAIN or grad and t.requires_grad:
            return False
    return True


_PLAIN = (torch.Tensor, torch.nn.Parameter)
_forward_ad = torch.autograd.forward_ad
_stack = torch._C._functorch.peek_interpreter_stack
_modes = torch._C._len_torch_dispatch_stack
_tracing = torch._C._get_tracing_state


def _plain_bf16(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Matrices whose rows the kernels can load 16 bytes at a time."""
    if not (x.is_cuda and x.dtype == w.dtype == torch.bfloat16
            and unrecorded(x, w) and x.dim() == w.dim() == 2):
        return False
    (a, b), (c, d) = x.stride(), w.stride()
    return b == 1 and d == 1 and a % 8 == 0 and c % 8 == 0 \
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0


MOST_ROWS = 512         # of a product that a kernel here takes


def _wave_gemm(M: int, N: int, K: int):
    """Tiles of 64 rows where those of 64 or 128 outputs are one workgroup a
    compute unit, or nearly: N of 11264 to 16384 and of 22528 to 32768.  Against
    the kernel of few rows or the library, us, x and w from memory: 32768 x 4096 1 row
    44.3 45.9, 16 47.3 46.0, 24 68 45, 64 66 47; 32768 x 2048 1 row 24.6 25.5, 32 29
    26, 64 38 26.5; 14272 x 3072 23 rows 20.5 18.2; 23744 x 4096 39 rows 47 35; 26112 x
    3072 6 rows 45 28; 60 random sizes, over the kernel of few rows 0.98 up to 4 rows,
    0.88 of 8 and 16.  Beyond 64 rows the library is as fast (96 of 32768 x 4096 63 60,
    128 64 65), and so it is with fewer or more tiles (10 of 7808 x 4096 17 21; 2 of
    39104 x 4096 59 64)."""
    if not 1 <= M <= 64 or K == 0 or K % 128 or N % 4:
        return None
    for bn in (64, 128):
        if 176 <= -(-N // bn) <= 256:
            return 64, bn, 1
    return None


def _full(tiles: int) -> float:
    """How full the units are over all waves of these."""
    return tiles / (-(-tiles // 256) * 256)


def _waves_gemm(M: int, N: int, K: int):
    """Tiles of 64 rows by 64 or 128 outputs where they are half a wave or more of one
    workgroup a compute unit, or several waves, against the kernel of few rows and the
    library; or that kernel, "rows", which reads whole lines since. 130 random sizes,
    time over what was there: 9153 to 11264 and 16385 to 22528 outputs 0.85 (4 of
    10628 x 3328 20 17; 16 of 10168 x 4224 34 19; 64 of 18736 x 896 15 11; 32 of 10008
    x 5120 26 27); several waves and up to 16 rows 0.87, wide tiles but where narrow
    ones fill the units better (1 of 128256 x 4096 185 163, 2 of 144224 x 2304 132
    113, 2 of 49448 x 3456 62 59), 17 to 32 rows 0.85 (128256 x 4096 201 172), 33 to
    64 with up to 4096 columns 0.80 (64 of 128256 x 4096 215 183). Left are 257 to 384
    wide tiles, which are nearly one wave more than needed, and narrow ones that fill
    no wave either (1.0 to 1.13); few columns for few rows (1 of 100164 x 640 28 30);
    long ones for many rows (62 of 58064 x 7296 156 161). The kernel of few rows in
    place of these tiles, up to 4 rows of 1152 to 5120 columns: 150 sizes 0.93 (1 of
    9600 x 4096 19.1 16.3, of 128256 x 4096 165 159, 2 of 100352 x 2048 77 66; worst 4
    of 256000 x 2048 162 172); 8 rows 0.89 to 1.2, longer columns 0.78 to 1.14,
    shorter ones 0.9 to 1.3."""
    tile = _several_waves(M, N, K)
    return "rows" if tile and M <= 4 and 1152 <= K <= 5120 else tile


def _several_waves(M: int, N: int, K: int):
    if not 1 <= M <= 64 or not 640 <= K <= 16384 or K % 128 or N % 4 \
            or N >= 1 << 24:        # outputs that the tiles count
        return None
    narrow, wide = -(-N // 64), -(-N // 128)
    if 144 <= narrow < 176:
        return 64, 64, 1
    if 128 < wide < 176:
        return 64, 128, 1
    if wide > 384 and (
            K >= 896 if M <= 16 else
            wide > 512 or _full(wide) >= 0.78 if M <= 32 else
            K <= 4096 and wide >= 500 and _full(wide) >= 0.75):
        return (64, 64, 1) if M <= 16 and _full(narrow) > _full(wide) + 0.08 \
            else (64, 128, 1)
    if 256 < wide <= 384 and M <= 16 and K >= 1152 and _full(narrow) >= 0.78:
        return 64, 64, 1
    return None


def _wave_of_rows(M: int, N: int, K: int):
    """Tiles of 64 x 64 for 65 to 192 rows where they are 144 to 256, so that every
    unit has at most one, on each of the 8 dies (of one tile of w all go to the same:
    3 tiles of rows and 84 of outputs are 252, but 33 on some).  250 random sizes, time
    over the library's: 2 tiles of rows, K of 384 to 1024 0.72, to 2304 0.9 (2 of 100
    more than 3 % slower), beyond 1.02; 3 0.73, beyond 2304 1.06 and more for every
    second one.  192 rows of 3072 x 2048 22 -> 12.6 us, 129 12.6 -> 11.1; decode steps
    of 8 layers with that product, 130 rows 964 -> 869 us, 192 1037 -> 939.  More rows
    gain in some steps and lose in others (256 1049 -> 1011, a prompt of 256 758
    766)."""
    if not 64 < M <= 192 or K % 128 or N % 4 or not 384 <= K <= 2304:
        return None
    mt, nt = -(-M // 64), -(-N // 64)
    return (64, 64, 1) if mt * nt >= 144 and -(-nt // 8) * mt <= 32 else None


def _wave_of_longer_rows(M: int, N: int, K: int):
    """The same tiles for 65 to 128 rows and longer columns where they are at least 176
    and the product would be the library's.  Random sizes, time over that: K up to 4608
    0.92 (66 rows of 7168 x 4096 24.6 -> 20.2 us), but of 97 to 128 rows up to 3712
    columns 1.03 in 62, up to 1.32 (125 of 6032 x 2560 13.7 17.0); longer ones every
    seventh slower, up to 1.11; fewer tiles 1.05 to 1.2.  In decode steps, a layer, 5632 x
    2560 to 8192 x 4608, 66 to 128 rows 1 to 8 us less.  In place of parts of 128 x 128 and
    the pass that adds them up, up to 6528 outputs from 4096 columns on, a product is 1 us
    faster by itself and a layer 0 to 4 us slower (8 layers with 6144 x 4096, 66 rows 1114
    -> 1128, 96 1143 1173, 128 1306 1330): they stay."""
    if not 64 < M <= 128 or K % 128 or N % 4 \
            or not (2304 if M <= 96 else 3712) < K <= 4608:
        return None
    nt = -(-N // 64)
    return (64, 64, 1) if 88 <= nt <= 128 else None


@lru_cache(maxsize=1 << 14)
def _route(M: int, N: int, K: int, parts: bool):
    """How x w^T of these sizes is formed: "rows", (rows, outputs of a tile, parts
    of K) or None, the library.  Kept, for the rules take as long as a launch: a
    step of small prompts, which is not captured, waits for the host."""
    if K >= 1 << 24:                # the kernels' chunks are counted in 32 bits
        return None
    wave = _wave_gemm(M, N, K) or _waves_gemm(M, N, K)
    if wave is not None:
        return wave
    if _rows_gemm_sizes(M, N, K) and _native().gemm_rows_fits(M, K):
        return "rows"
    return _less_padding(M, N, K, _split_gemm(M, N, K)) \
        or (_summed_gemm(M, N, K) or _few_parts(M, N, K) if parts
            else _wave_of_longer_rows(M, N, K)) \
        or _wave_of_rows(M, N, K)


def _rows_gemm_sizes(M: int, N: int, K: int) -> bool:
    """Measured at 1 to 64 rows, K of 256 to 4096 and N of 256 to 160000, 40000
    random sizes (time of the kernel over the library's, means of a class).  Up
    to 4096 outputs 0.53 to 0.84, but for more than 32 rows with K of 1280
    (1.0).  Beyond, the tiles of 16, 12 or 8 rows of w have to divide evenly
    over the 256 compute units (4608 x 2048, where the busiest has 1.33 times
    its share, is at 0.57 for one row and 0.71 for 16).  The loads of a step
    cover 2048 columns: K of 2048 is at 0.5 to 1.0 for all N, K of 4096 at 0.7 to 0.9 but
    for 6657 to 8192 outputs (1.05) and a head of 128256 with 16 rows (1.1).
    For other K the library is faster at 40961 to 65536 outputs (1.06 to 1.3);
    beyond, for up to 16 rows with K up to 1024 (0.94 to 1.26) and more with
    K up to 512 or beyond 3072 (1.0 to 1.3); below, for 17 to 32 rows with K
    beyond 1024 (0.93 to 1.16), for 33 to 64 with more than 12288 outputs (0.96
    to 1.6), for 32769 outputs and more with K up to 512 (1.0 to 1.8), and for
    6145 to 8191 outputs with K beyond 2048 (0.9 to 1.0 for one row, 0.98 to
    1.13 for 8 and 16).  2 to 6 of 100 sizes that are taken are more than 3 %
    slower than the library, where it has a tile that fits them."""
    if not 1 <= M <= 64 or K > 4096 or K % 8 or N % 4 or N * K < 1 << 20:
        return False
    if N <= 4096:
        return M <= 32 or not 1024 < K <= 1280
    most = min(-(-N // (256 * r)) * r
               for r in ((16, 12, 8) if M <= 16 else (16,)))
    if most * 256 > N * (1.34 if M <= 16 else 1.05):
        return False
    if K % 2048 == 0:
        return K == 2048 or not (6144 < N <= 8192 and M > 4
                                 or N > 65536 and M > 8)
    if M > 32:
        return K <= 1024 and N <= 12288
    if N > 65536:
        return 1024 < K if M <= 16 else K <= 3072 and (K > 512 or M <= 24)
    if N > (32768 if K <= 512 else 40960):
        return False
    if M > 16:
        return K <= 1024 or K < 2048 and N <= 20480
    return K < 2048 or M <= 4 or not 6144 < N < 8192


def _split_gemm(M: int, N: int, K: int):
    """(rows, outputs of a tile, parts of K) where csrc/gemm_split.hip is
    faster than the library, else None: products whose tiles, times the parts,
    are one workgroup a compute unit or less on each of the 8 dies (3 tiles of
    rows, 21 of outputs and 4 parts are 252, but 33 on some dies: 384 rows of
    2688 x 7552 took 47 us, the library 37).  Measured at 17 to 512 rows, N of
    512 to 9000 and K of 4096 to 20000: 0.67 of the library's time on average,
    and more than 3 % slower at 1 of 100 sizes.  Few parts gain less than the
    library's tiles up to 128 rows and from 257 on (us, library and kernel: 8192 x
    8192, 4 parts, 64 rows 33 43; 5120 x 8192, 3 parts, 320 rows 49 54).  From
    257 rows on short rows gain little or nothing (3072 x 6144, 320 rows 28 30;
    4096 x 6144 37 36, 512 rows 44 42).  Below 14M weights it is the faster one
    from K of 5120 on (2048 x 6144, 64 rows 19.5 12.3, 256 23 20) and about even
    with K of 4096 (2048 x 4096, 96 rows 12.7 12.6, 128 12.7 14.9); all these
    are left to the library.  So are 257 to 320 rows of up to 3264 outputs in
    tall tiles, K up to 12288 (3072 x 8192, 288 rows 34 38; 3136 x 7680, 257
    rows 32 37), 129 to 144 rows of more than 6528 outputs (7168 x 7168 42 45;
    6400 x 6400 at 0.68), and up to 32 rows where those of w lie a multiple of
    32 KB apart (4096 x 16384 31 42).  Narrow tiles where K is short and they
    fill as many units.
    129 to 256 rows in one tile, which loads three quarters of what two do, where
    that saves more than twice the parts cost: 120 sizes of K from 4608 to 20480,
    over what was there 0.86 with 4 or 5 parts (256 of 5648 x 7552 45 37, 192 of 7152
    x 5376 33 31), 0.92 with 6 or 7 of at least 8960 columns (189 of 4616 x 14464 52
    48) and with 8 of 15360 and up to 4 in tiles of 128, 0.96 to 1.15 else (256 of
    4096 x 14336 in a decode step even); with 2 or 3, against the library, 0.82 (256
    of 10112 x 4480 51 39, of 11168 x 7424 85 67; 163 of 15136 x 6656 65 65).  All of
    these in 50 other sizes, with x from memory, 0.83, the worst 1.03 (172 of 10576 x
    4352)."""
    if not 16 < M <= 512 or K < (4096 if M <= 256 else 7168) or K % 128 \
            or N % 4 or N * K < 14 << 20:
        return None
    if M <= 32 and K % 16384 == 0 and N >= 3072 \
            or 128 < M <= 144 and N > 6528 and K <= 16384:
        return None

    nt = -(-N // 128)
    if 128 < M <= 256 and nt <= 128:
        tall = min(8, 256 // nt)
        if K >= (6784 if tall == 2 else 4096 if tall == 3 else
                 4608 if tall <= 5 else 8960 if tall <= 7 else 15360) \
                and 128 // nt <= 4:
            return 256, 128, tall

    def parts(bm, bn):
        mt, nt = -(-M // bm), -(-N // bn)
        die = 32 // mt * 8          # tiles of outputs and parts on all dies
        return min(8, die // nt), mt * nt

    wide, tiles = parts(128, 128)
    if wide < (5 if M <= 128 else 2 if M <= 256 else 4):
        tall, _ = parts(256, 128)
        return (256, 128, tall) if M > 256 and tall >= 4 \
            and (M > 320 or N > 3264 or K > 12288) else None
    narrow, more = parts(128, 64)
    if M <= 256 and K < 8192 and more * narrow >= tiles * wide:
        return 128, 64, narrow
    return 128, 128, wide


def _less_padding(M: int, N: int, K: int, split):
    """Narrow tiles of 64 rows where those are enough: 17 rows of 2048 x 7168 8.2
    -> 8.0 us, 32 of 4096 x 4096 9.2 -> 8.7, 64 9.9 -> 9.5; the same bits.  In place of
    tiles of 128 x 128, in parts of their own, N of 1088 to 5440 and K of 4352 to 28672,
    with the norm or without: 5 parts and more 0.80 of the time (48 of 3072 x 8192 20.3
    -> 18.1 us, 33 of 2560 x 10240 19.9 16.9, 24 of 1344 x 19456 24 17; none slower).  4
    up to 18432 columns, or 12288 of more than 48 rows, 0.94 in 83 (40 of 4096 x 16384
    45 30, 24 of 4096 x 8192 21.0 20.0), beyond 1.0 in 78, up to 1.24; 3 up to 12288, or
    8192, 0.97 in 39 (32 of 4608 x 8192 24.2 21.5), beyond 1.04 in 166, up to 1.29; 2
    1.06.  2 of the 122 that are taken are more than 3 % slower."""
    if not split or M > 64 or split[0] != 128:
        return split
    if split[1] == 64:
        return 64, 64, split[2]
    narrow = min(8, 256 // -(-N // 64))
    most = (8192, 12288) if M > 48 else (12288, 18432)
    return (64, 64, narrow) if narrow >= 5 \
        or narrow >= 3 and K <= most[narrow - 3] else split


def _few_parts(M: int, N: int, K: int):
    """Two or three parts of one tile of up to 64 rows, where the norm adds them up and
    no other rule has a kernel.  N of 4160 to 8192 and K of 4224 to 28672, with the norm,
    over the library's time: 2 parts 0.72 in 66, none above 0.96 (1 row of 8192 x 28672
    94 78 us, 12 of 7168 x 18432 114 51, 1 of 6656 x 17920 92 47, 8 of 8192 x 8192 34.4
    30.5), 3 0.9 (4 of 5120 x 5120 18.2 16.7, 1 17.7 16.6), but up to 5120 columns, of
    multiples of 256, and up to 4992 outputs 1.1 and more for every second size (2 of
    4608 x 4608 13.4 15.1, 1 of 4168 x 5120 13.3 15.6, 1 of 4864 x 5120 0.97); those are
    the library's, and so are 4096 columns and fewer (16 of 8192 x 4096 20 22.5)."""
    if not 1 <= M <= 64 or K % 128 or N % 8 or not 0 < N <= 8192 \
            or not 4096 < K <= 28672:
        return None
    split = 256 // -(-N // 64)
    if split == 3 and K <= 5120 and K % 256 == 0 and N <= 4992:
        return None
    return (64, 64, split) if 2 <= split <= 3 else None


def _summed_gemm(M: int, N: int, K: int):
    """As _split_gemm, for more sizes, where the norm adds up the parts.  Measured
    with the norm.  1 to 16 rows, K of 5120 to 20000 and N of 64 to 8192 in 400
    random sizes: with 5 parts or more (N up to 3264) 0.62 of the library's time on
    average (9 rows of 512 x 5632 9.6 9.1, 1 of 2048 x 7168 14.3 11.8, 15 of 3072 x
    5120 13.7 12.8; the slowest 5 of 3072 x 16384 26.6 28.1).  With 3 or 4 about even
    up to 8192 columns (2 of 4096 x 7168 16.7 17.4, 10 of 5168 x 7168 23.2 21.4) but
    where K is no multiple of 512 (8 of 4392 x 6784 31 19), beyond 0.8 (1 of 4096 x
    14336 28.8 27.5, 9 of 4096 x 11264 24.1 24.2), and slower where rows lie a
    multiple of 16 KB apart (8 of 4096 x 8192 18.7 22.9).  33 to 128 rows with K of
    1024 to 4096 and less than 14M weights: 0.87 in 65 sizes, none slower by 3 % (48
    rows of 2048 x 2048 11.0 8.9 us, 64 of 4096 x 2560 13.4 12.5, 78 of 3200 x 3584
    23 14).  257 to 512 rows with K from 5120 on, or 4096 in tiles of 128 rows: 0.92
    in 40 (480 of 4096 x 4096 33 32, 395 of 5120 x 7168 60 51, 298 of 3968 x 6144 40
    35, 454 of 4224 x 11008 93 68).  Two parts of tall tiles are even (452 of 5504 x
    8192 65 70, 379 of 7168 x 14336 119 116) but with long columns and full tiles, 0.86
    in 8 of 8704 and more (512 of 6504 x 10496 100 84, 454 of 6336 x 8192 66 67)."""
    if K % 128 or N % 8 or not 0 < N <= 8192:
        return None
    if M <= 16 and K >= 5120 and N * K >= 2 << 20:
        split = min(6, 256 // -(-N // 64), K // 1024)
        return (64, 64, split) if split >= 5 or split >= 3 and K % 8192 and (
            K > 8192 or K % 512) else None
    if 32 < M <= 128 and 1024 <= K <= 4096 and 1 << 20 <= N * K < 14 << 20:
        split = min(8, 256 // (-(-M // 64) * -(-N // 64)), K // 512)
        return (64, 64, split) if split > 1 else None
    if 256 < M <= 512 and K >= 4096:
        mt, nt = -(-M // 128), -(-N // 128)
        wide, tall = 32 // mt * 8 // nt, min(8, 128 // nt)
        if wide >= 2 and (M > 384 and tall < 3 or K < 5120 or
                          M <= 384 and mt * wide >= 1.6 * tall):
            return 128, 128, min(8, wide)
        if tall >= (2 if K >= 8704 else 3) and K >= 5120:
            return 256, 128, tall
    return None


# Tiles of csrc/gemm_wide.hip, 32 * high rows by bn outputs: us of a wave of 256 and of
# 64 columns of it, least squares over 2900 random sizes (6 % off on average).
_WIDE_TIMES = {(4, 128): (0.0, 0.60), (5, 128): (0.5, 0.65),
               (6, 128): (1.8, 0.68), (7, 128): (2.6, 0.75),
               (8, 128): (3.1, 0.84), (4, 256): (3.6, 0.80),
               (5, 256): (1.8, 0.96), (6, 256): (2.6, 1.08),
               (7, 256): (4.5, 1.21), (8, 256): (5.3, 1.40)}


def _wide_tile(M: int, N: int, K: int, parts=(1,)):
    """(us, high, bn, parts of K, tiles) of the tiles that take the least time: even
    tiles of up to 256 rows, or one more of them if they are several.  Parts are floats
    that the norm reads."""
    best, least = None, -(-M // 256)
    for mt in (least, least + (least > 1)):
        high = -(-M // (mt * 32))
        for bn in (128, 256):
            if (high, bn) not in _WIDE_TIMES:
                continue
            fixed, chunk = _WIDE_TIMES[high, bn]
            for split in parts:
                tiles = -(-M // (high * 32)) * -(-N // bn) * split
                if split > 1 and (tiles > 256 or K < 256 * split):
                    continue
                us = -(-tiles // 256) * (fixed + chunk * K / 64 / split) \
                    + M * N * (4 if split == 1 else 8 * split) / 5e6
                if best is None or us < best[0]:
                    best = us, high, bn, split, tiles
    return best


@lru_cache(maxsize=1 << 14)
def _wide_gated(M: int, N: int, K: int):
    """(high, bn) where csrc/gemm_wide.hip forms silu(gate) * up of more than 256
    rows faster than what was there, mostly the library's product and a pass.  Random
    sizes, N of 6000 to 36000, at 0.7 PFLOP/s and more by the tiles' times, time over
    that: up to 1200 rows 0.88 in 186 (880 of 28672 x 4096 197 187 us, 512 109 109, but
    6 less a layer in the step, 512 of 14336 x 2048 36 35), 8 of them more than 3 %
    slower, up to 8 %, and 769 and more of them of over 5376 columns 0.93 in 74, but 19
    slower, up to 14 % (1192 of 16384 x 5888 210 239): those are the library's.  More
    rows of up to 3072 columns 0.86 in 20 (2600 of 14336 x 2048 181 143), of longer ones
    0.95, but every fourth slower, by up to 10 % (8192 of 28672 x 4096 1335 1400): those
    are the library's too."""
    if not 256 < M < 1 << 20 or K < 1024 or K % 64 or N % 16 \
            or not 6000 <= N < 1 << 17 \
            or K > (8192 if M <= 768 else 5376 if M <= 1200 else 3072):
        return None
    us, high, bn, _, _ = _wide_tile(M, N, K)
    return (high, bn) if 2e-9 * M * N * K / us >= 0.7 else None


@lru_cache(maxsize=1 << 14)
def _wide_parts(M: int, N: int, K: int):
    """(high, bn, parts) where csrc/gemm_wide.hip and the norm that adds up its parts
    are faster than what was there and the norm.  Random sizes, x and w from memory,
    time over that: 10240 columns and more, up to 1400 rows 0.69 in 97 (262 rows of
    4096 x 14336 64 52 us, 600 121 80, 1000 145 114, 1268 165 146; the worst 1154 of 6336
    x 15360 even), but 1.09 for tiles that fill no wave and 1.10 in 45 for one part of
    tiles of 256 outputs, which are 180 to 217 (1114 of 8144 x 12928 231 252); from 4608
    on 513 to 1024 rows 0.90 in 57 (the worst 989 of 8032 x 4992 89 92).  Shorter ones
    are slower (up to 2560 columns and 4096 outputs, 513 to 1024 rows, 1.14 in 93, 630 of
    1768 x 2048 17.6 21.1), and so are more rows (1.0).
    129 to 256 rows of 10240 columns and more, one tile of rows and more than 192 in all,
    0.65 (135 rows of 4096 x 14336 47 40 us, 248 52 50); decode steps of 140, 200 and 256
    rows, 8 layers, 1 % less.  Fewer rows are as fast in the step (100 1730 1738), fewer
    tiles slower (200 of 2048 x 7168 17 21)."""
    if K % 64 or N % 8 or not 1024 <= N <= 8192 or not 4608 <= K <= 20480 \
            or not 128 < M <= (1400 if K >= 10240 else 1024):
        return None
    _, high, bn, split, tiles = _wide_tile(M, N, K, (1, 2, 3, 4, 5, 6, 7, 8))
    if M <= 256:
        fits = tiles > 192 and K >= 10240
    elif M <= 512:
        fits = 176 <= tiles <= 256 and K >= 10240 and N >= 1536
    else:
        fits = 176 <= tiles <= 256 and (split > 1 or bn == 128)
    return (high, bn, split) if fits else None


@lru_cache(maxsize=1 << 14)
def _wide_long(M: int, N: int, K: int):
    """(high, bn, 1) for long columns where 256 x 256 tiles are two or three waves of
    which the last is neither nearly empty nor full.  The library has two kinds of
    tiles, of 0.65 to 1.1 PFLOP/s and of 1.2 to 1.5; here it is 1.1 to 1.35.  N from 2048
    to 8192, K from 10240 to 32768, time over the library's: two waves 0.73 in 85 (7411
    rows of 4096 x 14336 1006 647 us, 5888 of 5120 x 13824 974 629), four of them more
    than 3 % slower, by up to 15 % (7425 of 4096 x 11008), three 0.87 in 81, three
    slower, by up to 12 % (5889 of 7168 x 18432), but multiples of 64 tiles, for which
    it mostly has the better ones, 1.04 in two waves; more waves 1.0 in 20, every second
    one slower.  With up to 10240 columns it has 1.3 to 1.55."""
    if not 1024 < M <= 16384 or not 10240 <= K <= 1 << 15 or K % 64 or N % 8 \
            or not 2048 <= N <= 8192:
        return None
    tiles = -(-M // 256) * -(-N // 256)
    if not 256 < tiles <= 768 or tiles % 64 == 0 \
            or not 0.8 <= _full(tiles) < 0.96:
        return None
    _, high, bn, _, _ = _wide_tile(M, N, K)
    return high, bn, 1


def _near(x: torch.Tensor, w: torch.Tensor, bm: int, bn: int) -> bool:
    """32 bits of offset reach the rows of a tile of bm by bn from its first."""
    return all(((min(t.shape[0], rows) - 1) * t.stride(0) + t.shape[1])
               * t.itemsize < 0xfffffff0 for t, rows in ((x, bm), (w, bn)))


def _product(x: torch.Tensor, w: torch.Tensor, parts: bool, plain: bool):
    """x w^T for w [N, K]; with `parts` as Parts where it is formed so.  plain:
    what _plain_bf16 says, which looks at the sizes of no traced tensor."""
    M, N = x.shape[0], w.shape[0]
    wide = plain and M > 128 and (parts and _wide_parts(M, *w.shape)
                                 or _wide_long(M, *w.shape))
    if wide and _near(x, w, wide[0] * 32, wide[1]):
        high, bn, split = wide
        part = torch.empty(split, M, N, dtype=torch.float32,
                           device=x.device) if split > 1 else None
        out = None if part is not None else \
            torch.empty(M, N, dtype=x.dtype, device=x.device)
        _native().gemm_wide(out, x, w, part, high, bn, split)
        return out if part is None else Parts(part)
    route = _route(M, *w.shape, parts) if plain and M <= MOST_ROWS else None
    if route is None or route != "rows" and not _near(x, w, *route[:2]):
        return x @ w.t()
    if route == "rows":
        out = torch.empty(M, N, dtype=x.dtype, device=x.device)
        _native().gemm_rows(out, x, w)
        return out
    part = torch.empty(route[2], M, N, dtype=torch.float32,
                       device=x.device) if route[2] > 1 else None
    if parts and part is not None and N % 8 == 0 and N <= 8192:
        _native().gemm_split(None, x, w, part, *route)
        return Parts(part)
    out = torch.empty(M, N, dtype=x.dtype, device=x.device)
    _native().gemm_split(out, x, w, part, *route)
    return out


def linear_parts(x: torch.Tensor, w: torch.Tensor):
    """x w^T for w [N, K], as Parts where it is formed in parts of K."""
    return _product(x, w, True, _plain_bf16(x, w))


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x w^T for w [N, K]."""
    return _product(x, w, False, _plain_bf16(x, w))


@lru_cache(maxsize=1 << 14)
def _gated_tile(M: int, N: int, K: int):
    """(rows, rows of w of a tile) where csrc/gemm_split.hip forms silu(gate) *
    up of x w^T faster than a product and an activation, else None: the smallest
    tiles that are one workgroup a compute unit or less.  Measured at 1 to 256
    rows, N of 2048 to 57344 and K of 512 to 8192: 0.78 of both on average where
    it is taken (us, x and w from memory: 28672 x 4096 1 row 64 41, 8 rows 65 41, 17
    52 41, 32 52 41, 64 53 42, 128 61 53; 14336 x 2048 1 row 19 13, 16 18 12, 32 18 13,
    64 20 15, 128 23 19, 192 30 23, 256 33 24).
    More tiles take a second wave (192 rows of 28672 x 4096 67 73) but for 17 to
    64 rows, where the library has no better tile (29 rows of 38400 x 6144 124
    96; 6 of 52736 x 1536 36 38).  Few tiles with long rows leave the chip idle (23 rows of 2048 x 3072
    10 13), and more than 64 rows of more than 4096 columns gain nothing (71 of
    6144 x 5120 22.5 22.8, 119 of 5632 x 5120 25 27)."""
    if not 1 <= M <= 256 or K == 0 or K % 128 or N % 16 \
            or M > 64 and K > 4096 or max(N, K) >= 1 << 24:
        return None
    for bm, bn in ((64, 64), (64, 128)) if M <= 64 \
            else ((64, 64), (128, 64), (128, 128)):
        tiles = -(-M // bm) * -(-N // bn)
        if tiles <= 256:
            least = 128 if K > 2048 else 72 if M <= 16 else \
                64 if K > 1024 else 40
            return (bm, bn) if tiles >= least else None
    return (64, 64) if 16 < M <= 64 else None


@lru_cache(maxsize=1 << 14)
def _gated_wave(M: int, N: int, K: int):
    """(256, 128) where those tiles of silu(gate) * up are one workgroup a compute
    unit, and half of the units or more have one, for 129 to 512 rows.  The product
    alone takes as long as the library's, so what is gained is the activation's
    pass, and with few columns more.  Measured in 210 random sizes, time over that
    of both: K up to 4608 0.80 in 80 of 130 to 256 tiles, none above 0.99 (256 of
    28672 x 4096 79 69 us, 512 of 14336 x 1664 36.1 27.4, 129 of 20192 x 2816 45.8
    40.9); up to 7168 with 208 tiles and more 0.93 (512 of 14848 x 6912 110 99, 132
    of 28032 x 5120 77.9 79.3), with fewer 1.03; beyond 1.02.  Fewer tiles lose with
    up to 256 rows, where narrower ones fit, and beyond, but for up to 1024 columns
    (376 of 7392 x 640 16.6 13.1; 467 of 8192 x 3584 42 47)."""
    if not 128 < M <= MOST_ROWS or K == 0 or K % 128 or N % 16 \
            or max(N, K) >= 1 << 24:
        return None
    tiles = -(-M // 256) * -(-N // 128)
    if 128 < tiles <= 256 and K <= (7168 if tiles >= 208 else 4608) \
            or M > 256 and 96 <= tiles <= 128 and K <= 1024:
        return 256, 128
    return None


def gated_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu_mul of x w^T, w the gate's rows and then the up rows."""
    plain = _plain_bf16(x, w)
    sizes = (x.shape[0], *w.shape) if plain else None
    wide = plain and _wide_gated(*sizes)
    if wide and _near(x, w, wide[0] * 32, w.shape[0] // 2 + 128):
        out = torch.empty(x.shape[0], w.shape[0] // 2, dtype=x.dtype,
                          device=x.device)
        _native().gemm_wide(out, x, w, None, *wide, gated=True)
        return out
    if plain and x.shape[0] <= MOST_ROWS:
        tile = _gated_tile(*sizes) or _gated_wave(*sizes)
        if tile is not None and _near(x, w, *tile) \
                and w.stride(0) * (w.shape[0] + 256) < 1 << 32:
            out = torch.empty(x.shape[0], w.shape[0] // 2, dtype=x.dtype,
                              device=x.device)
            _native().gemm_split(out, x, w, None, *tile, 1, gated=True)
            return out
    return silu_mul(_product(x, w, False, plain))


class QTensor(NamedTuple):
    """Per-token-scaled fp8 activation: data e4m3fn [T,K], scale fp32 [T].

    Produced on GPU by the fused quant kernels (csrc/quant.hip) so fp8
    GEMM inputs never take an extra elementwise pass; consumed by the TP
    linear layers via linear_q."""

    data: torch.Tensor
    scale: torch.Tensor


class PaddedQ(QTensor):
    """Rows of a captured step: those of a negative slot are padding."""

    slots: Optional[torch.Tensor] = None


@lru_cache(maxsize=1 << 14)
def _tiles_q(M: int, N: int, K: int, parts: bool):
    """(rows, outputs of a tile, parts of K) where csrc/gemm_split.hip is
    faster than the library for x e4m3 [M, K] and w e4m3 [N, K], else None.
    With `parts` their sum costs little, for the norm that follows forms it.

    Measured at 1 to 128 rows, N of 1024 to 40000 and K of 1024 to 14336 in 400
    random sizes: 0.8 of the library's time on average, and more than 3 % slower
    at 3 of 100.  Tiles of 64 x 64 that fill three quarters of the compute
    units need no parts (16 rows of 28672 x 4096 33.8 -> 24.5 us, 64 of 14336 x
    2048 14.3 -> 11.0), and more than one wave of them are one wave of twice the
    width (64 rows of 28672 x 4096 31.1 -> 25.7, 64 wide 28.8; 16 of 21184 x 4096
    28.9 20.4 21.7), but not with a second wave that is nearly full and few rows
    (32 of 28672 x 4096 25.8 and 25.0), or short rows (64 of 23232 x 1024 11.1
    10.9).  With K beyond 4096 in tiles of 64, beyond 6144 in wider ones, the
    library catches up from 17 rows on (20 rows of 12768 x 6144 18.1 18.0; 64 of
    19936 x 6144 34.0 34.4 wide, 48 of 24336 47.7 33.3), with more than 32768
    outputs for any (16 rows of 35312 x 6144 48 57).  Fewer tiles are
    divided into parts of 1365 columns and more, about one workgroup a unit (64
    rows of 4096 x 14336 with the norm 30.6 -> 21.5, of 2048 x 7168 16.3 ->
    12.8), or made half as wide (6144 x 4096 13.7 -> 12.3, 3072 x 2048 9.1 ->
    6.4).  Where another kernel adds up the parts they gain with 8192 columns,
    or with few rows (1 of 3600 x 5120 14.0 -> 9.2; 21 of 6032 x 5120 11.7 13.0).
    Beyond 64 rows half as many tiles lie beside each other: long rows only with
    the norm (128 of 4096 x 14336 44 -> 28), 2048 x 7168 is even (14.0 13.7).
    Beyond 128 rows there is no gain (200 of 4096 x 4096 17.1 17.2)."""
    if not 1 <= M <= 128 or K % 256 or N % 4 or N * K < 1 << 22 \
            or K >= 1 << 24:
        return None
    tiles = -(-M // 64) * -(-N // 64)
    few = M <= 16
    if tiles >= 192:
        wide = 256 < tiles <= 512 and K >= 2048 and (tiles <= 384 or M > 32)
        return (64, 128 if wide else 64, 1) \
            if N <= (32768 if M <= 64 else 20480) and (
                few or K <= 2048 or K <= 4096 and (M <= 64 or N <= 8192)
                or wide and M <= 64 and K <= 6144) else None
    split = min(8, max(2, K // 1365), 256 // tiles)
    if M > 64 and K > 4096 and (K < 8192 or split == 1 or not parts):
        return None
    if parts and split > 1:
        return 64, 64, split
    if K > 4096:
        return (64, 64, max(2, split)) \
            if tiles <= 96 and (few or K >= 8192) else None
    if K > 2048 and tiles < (64 if M <= 64 else 128):
        return (64, 64, min(8, 256 // tiles)) if few else None
    return (64, 32, 1) if tiles <= 128 else (64, 64, 1)


def _aligned_q(x: "QTensor", w: torch.Tensor, scale: torch.Tensor) -> bool:
    d, s = x
    return d.dtype == w.dtype == torch.float8_e4m3fn \
        and s.dtype == scale.dtype == torch.float32 \
        and s.is_contiguous() and scale.is_contiguous() \
        and scale.data_ptr() % 16 == 0 \
        and all(t.stride(1) == 1 and t.stride(0) % 16 == 0
                and t.data_ptr() % 16 == 0 for t in (d, w))


def _tiled_q(x: "QTensor", w: torch.Tensor, scale: torch.Tensor, parts: bool):
    """The tile of _tiles_q, or None."""
    tile = _tiles_q(x.data.shape[0], *w.shape, parts)
    return tile if tile is not None and _near(x.data, w, *tile[:2]) \
        and _aligned_q(x, w, scale) else None


@lru_cache(maxsize=1 << 14)
def _rows_q_sizes(M: int, N: int, K: int, parts: bool) -> bool:
    """Where csrc/gemm_rows.hip is faster for e4m3, which reads whole lines of w
    without a tile's padding: up to 32 rows that the library or the narrowest tiles
    took, and up to 16 in parts of up to 8192 columns that a kernel of their own would
    add up.  180 sizes, time over that of what was there: against the library 0.34 to
    0.98 (8 of 8880 x 14592 79 30, 16 of 1280 x 2304 7.0 4.5), tiles of 32 outputs
    0.64 to 0.92 (1 of 6144 x 4096 9.8 6.8, 16 11.1 8.9, 32 of 2048 x 2048 6.5 5.0; 38
    of 6112 x 2304 7.5 9.2), parts 0.63 to 0.99 (8 of 1760 x 3072 6.6 4.3; of longer
    ones up to 1.27).  Full waves of wider tiles are faster (16 of 14336 x 2048 8.8
    10.9), and so are parts that the norm adds up."""
    if not 1 <= M <= 32 or K % 16 or N % 4 or N * K < 1 << 19 or K > 1 << 17 \
            or N >= 1 << 24:        # not measured; the kernel counts to 2^31
        return False
    tile = _tiles_q(M, N, K, parts)
    return tile is None or tile[1] == 32 or (
        tile[2] > 1 and not parts and M <= 16 and K <= 8192)


def linear_q(x: "QTensor", w: torch.Tensor, scale: torch.Tensor,
             parts: bool = False):
    """x w^T of e4m3 with scales of the rows, bf16; with `parts` as Parts where
    it is formed in parts of K.  GPU."""
    # The host's time is what an eager step of small prompts waits for, so rows are
    # counted first.  But not those of a traced tensor, which a comparison would fix:
    # their number is no int, or only looks like one to what compiles.
    d, rows, tile = x.data, None, None
    if not torch.compiler.is_compiling() and d.dim() == w.dim() == 2:
        rows = d.shape[0]
    if type(rows) is int and rows <= 128 and d.is_cuda \
            and unrecorded(d, w, x.scale, scale):
        if rows <= 32 and d.shape[1] == w.shape[1] \
                and _rows_q_sizes(rows, *w.shape, parts) \
                and _aligned_q(x, w, scale) \
                and _native().gemm_rows_fits(rows, w.shape[1] // 2):
            out = torch.empty(rows, w.shape[0], dtype=torch.bfloat16,
                              device=w.device)
            _native().gemm_rows(out, d, w, x.scale, scale)
            return out
        tile = _tiled_q(x, w, scale, parts)
    if tile is None:
        return torch._scaled_mm(x.data, w.t(), scale_a=x.scale.unsqueeze(1),
                                scale_b=scale.unsqueeze(0),
                                out_dtype=torch.bfloat16)
    M, N = x.data.shape[0], w.shape[0]
    part = torch.empty(tile[2], M, N, dtype=torch.float32,
                       device=w.device) if tile[2] > 1 else None
    keep = parts and part is not None and N % 8 == 0 and N <= 8192
    out = None if keep else torch.empty(M, N, dtype=torch.bfloat16,
                                        device=w.device)
    _native().gemm_split(out, x.data, w, part, *tile, x.scale, scale)
    return Parts(part) if keep else out


def quant_fp8(x: torch.Tensor) -> QTensor:
    """[T,K] bf16 -> QTensor (GPU; row-per-workgroup amax+scale+pack)."""
    assert x.is_cuda
    T, K = x.shape
    out = torch.empty(T, K, dtype=torch.float8_e4m3fn, device=x.device)
    scales = torch.empty(T, dtype=torch.float32, device=x.device)
    _native().quant_fp8(out, scales, x)
    return QTensor(out, scales)


def fused_add_rmsnorm_q(x: torch.Tensor, residual: torch.Tensor,
                        weight: torch.Tensor, eps: float):
    """residual += x (in place); returns (QTensor of rmsnorm(residual)*w,
    residual).  GPU-only fused producer for the fp8 GEMM path."""
    if isinstance(x, Choices):
        x = _moe_sum(x)
    T, K = residual.shape
    out = torch.empty(T, K, dtype=torch.float8_e4m3fn, device=residual.device)
    scales = torch.empty(T, dtype=torch.float32, device=residual.device)
    if isinstance(x, Parts):
        _native().parts_add_rmsnorm_fp8(out, scales, x.data, residual, weight,
                                        eps)
        return QTensor(out, scales), residual
    assert x.is_cuda
    _native().fused_add_rmsnorm_fp8(out, scales, x, residual, weight, eps)
    return QTensor(out, scales), residual


def silu_mul_q(gate_up: torch.Tensor) -> QTensor:
    """silu(g)*u -> fp8 QTensor (GPU fused producer)."""
    assert gate_up.is_cuda
    i = gate_up.shape[-1] // 2
    out = torch.empty(*gate_up.shape[:-1], i, dtype=torch.float8_e4m3fn,
                      device=gate_up.device)
    scales = torch.empty(gate_up.shape[0], dtype=torch.float32,
                         device=gate_up.device)
    _native().silu_mul_fp8(out, scales, gate_up)
    return QTensor(out, scales)


MOE_BM = 256  # sorted-pair tile granularity of the MoE kernels (csrc/moe.hip)


def _moe_splitk(nblocks: int, nchunks: int, out_numel: int, dev):
    """Split-K degree + fp32 workspace for a launch of csrc/moe.hip, the
    grouped GEMM of large steps of the designs in ops/experts.py.

    A launch of a few more blocks than the 256 CUs have idles most of the
    chip in its second wave; splitting K into up to 8 segments (each must
    keep >= 3 k-chunks for the LDS ring and divide the chunk count)
    multiplies the block count back above ~4 per CU.  Shapes-only decision:
    hipGraph-capture-safe.
    HS_MOE_SPLITK forces a degree (0 = auto)."""
    forced = int(os.environ.get("HS_MOE_SPLITK", "0"))
    s = 1
    if forced and nblocks >= 1024:
        forced = 0          # forcing never touches saturated launches
    while (s < 8 and nchunks % (s * 2) == 0 and nchunks // (s * 2) >= 3
           and (nblocks * s < 1024 if not forced else s * 2 <= forced)):
        s *= 2
    if forced == 1:
        s = 1
    if s == 1:
        return 1, None
    return s, torch.empty(s * out_numel, dtype=torch.float32, device=dev)


def moe_router_takes(tokens: int, experts: int) -> bool:
    """Whether the router kernel, which reads the router's rows for every
    token, is faster than torch's product, softmax and selection (us, torch
    and kernel: 16 x 4096, 2048 tokens 70 25, 8192 111 86, 16384 182 186; 32 x
    2048, 4096 tokens 72 52, 6144 78 74, 8192 86 98; 64 x 4096, 192 tokens 51
    14, 1024 67 54, 1280 77 67, 2048 83 106, 8192 138 401; 64 x 2048, 1280 63
    52, 2048 69 80)."""
    return experts <= 64 and tokens <= (
        16384 if experts <= 16 else 6144 if experts <= 32 else 1280)


def moe_router(x, router: torch.Tensor, top: int,
               slots: Optional[torch.Tensor] = None):
    """(weights [T, top] float, expert ids [T, top] int32) of the rows of x, a
    bf16 tensor or a QTensor: the softmax over the chosen.  Rows of a negative slot
    (int64) choose none.  GPU."""
    data, scale = x if isinstance(x, QTensor) else (x, None)
    T = data.shape[0]
    weight = torch.empty(T, top, dtype=torch.float32, device=data.device)
    ids = torch.empty(T, top, dtype=torch.int32, device=data.device)
    _native().experts_router(weight, ids, data, scale, router, top, slots)
    return weight, ids


# Mean rows per expert up to which the kernels without a sort, and tiles of 64
# and 128 rows are taken (and 256 beyond).  64 leave room for the spread of the
# counts: a few rows more than a tile and an expert's weights are read twice, by
# workgroups that share their compute units with others.  Tiles of 256 are as high as
# their choices, so 128 are no faster from 80 on and 1.3 times as slow where an expert
# has more of them.  us on an MI355X without a sort, and in tiles of 64, 128, 256, sort
# included, and where the first experts are chosen 1.9 times as often as the last
#   8 experts of 14336 x 4096   1 row 280 342, 2 rows 430 447, 3 438 453, 5 450
#     449, 48 - 470 521 507, 56 - 589 526 527, 80 - 766 564 533, 100 - 804 580 575,
#     112 - 813 589 566, uneven 80 - 746 547 536, 112 - 898 723 568
#   16 of 2048 x 4096           1 row 86 106, 3 rows 133 141, 5 137 140, 48 -
#     145 152 164, 56 - 163 153 162, 80 - 197 163 169, 100 - 213 172 169, 112 - 235 199
#     176, uneven 80 - 206 165 169, 100 - 225 203 172
#   32 of 1024 x 2048           1 row 51 60, 3 rows 71 75, 5 77 75, 48 - 81 89
#     83, 56 - 101 91 84, 80 - 112 96 92, 100 - 114 101 93, uneven 100 - 129 121 98
#   64 of 1024 x 2048           1 row 86 97, 3 rows 131 135, 5 153 140, 48 - 145
#     170 161, 80 - 208 191 178, 100 - 234 202 183, uneven 100 - 253 228 183
# 256 over 128 in seven stacks, even and uneven, and e4m3 in four: 56 0.99 0.97 1.02, 80
# 0.97 0.97 0.99, 90 0.96 0.96 0.97, 100 0.96 0.87 0.98, 112 0.88 0.84 0.94; the worst
# from 90 on 16 of 3072 x 6144, 366 401, up to 80 16 of 2048 x 4096.
# Choices that are uneven are better in the next larger tiles where several experts
# have a little more than a tile: 190 tokens of 8 experts, 47.5 choices on average, us
# in tiles of 64, 128, 256, even 477 519 511, the first 1.5 times as often as the last
# 481 515 512, 2.3 times 566 514 514.
MOE_ROWS, MOE_ROWS_64, MOE_ROWS_128 = 2.9, 48, 80


def _moe_tile(T: int, K: int, E: int, least: int) -> int:
    mean = T * K / E
    if mean <= MOE_ROWS and least <= 16:
        return 16
    return 64 if mean <= MOE_ROWS_64 else 128 if mean <= MOE_ROWS_128 else 256


def _moe_sizes(E: int, H: int, I: int) -> None:
    """Refuses what the experts' kernels cannot take."""
    if E > 64 or H % 128 or I % 128:
        raise RuntimeError(f"moe: {E} experts of {I} x {H}: at most 64, and "
                           "sizes that are multiples of 128")


def _moe_sort(ids: torch.Tensor, E: int, H: int, I: int, bm: int):
    """(order, expert, place) of the choices `ids` [T, K], sorted in tiles of
    bm rows."""
    _moe_sizes(E, H, I)
    pairs = ids.numel()
    tiles = min(pairs, (pairs + E * (bm - 1)) // bm)
    i32 = lambda *s: torch.empty(*s, dtype=torch.int32, device=ids.device)
    order, expert, place = i32(tiles * bm), i32(tiles), i32(*ids.shape)
    _native().experts_sort(order, expert, place,
                           ids.reshape(-1).to(torch.int32), E, bm)
    return order, expert, place


def _moe_sum(c: Choices) -> torch.Tensor:
    y, place = c.data, c.place
    out = torch.empty(place.shape[0], y.shape[1], dtype=y.dtype,
                      device=y.device)
    _native().experts_sum(out, y, place, c.weights, None, None, None, None,
                          0.0)
    return out


def moe_ffn(x: torch.Tensor, w13: torch.Tensor, w2: torch.Tensor,
            weights: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
    """Grouped expert SwiGLU FFN (GPU, hipGraph-capture-safe).

    x [T,H]; w13 [E_local, 2I, H]; w2 [E_local, H, I]; weights [T,K] fp32/bf16
    routing weights; ids [T,K] LOCAL expert indices.  Token->expert sorting,
    the two grouped MFMA GEMMs and the weighted combine all run on-device
    with grids that depend only on (T, K, E) — no host sync, no dynamic
    shapes (MoE dispatch/combine + grouped GEMM).
    """
    if x.shape[0] == 0:
        return torch.empty_like(x)
    return _moe_sum(moe_choices(x, w13, w2, weights, ids))


def moe_choices(x: torch.Tensor, w13: torch.Tensor, w2: torch.Tensor,
                weights: torch.Tensor, ids: torch.Tensor) -> Choices:
    """moe_ffn of at least one token without its closing sum."""
    n = _native()
    (T, H), K, (E, _, I) = x.shape, ids.shape[1], w2.shape
    bm = _moe_tile(T, K, E, 16)
    if bm == 16:
        _moe_sizes(E, H, I)
        ids = ids.to(torch.int32).contiguous()
        place = torch.empty_like(ids)
        h = torch.empty(T * K, I, dtype=torch.bfloat16, device=x.device)
        y = torch.empty(T * K, H, dtype=torch.bfloat16, device=x.device)
        n.experts_few(True, h, place, x, w13, ids, K)
        n.experts_few(False, y, None, h, w2, ids, 1)
        return Choices(y, place, weights.float().contiguous())
    order, expert, place = _moe_sort(ids, E, H, I, bm)
    P = order.shape[0]
    h = torch.empty(P, I, dtype=torch.bfloat16, device=x.device)
    y = torch.empty(P, H, dtype=torch.bfloat16, device=x.device)
    n.experts_tiles(h, x, w13, None, None, order, expert, True, K, bm)
    n.experts_tiles(y, h, w2, None, None, order, expert, False, 0, bm)
    return Choices(y, place, weights.float().contiguous())


def moe_ffn_fp8(xq: "QTensor", w13q: torch.Tensor, w13s: torch.Tensor,
                w2q: torch.Tensor, w2s: torch.Tensor,
                weights: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
    """fp8 grouped expert FFN: e4m3fn activations (QTensor from the fused
    norm producer) x e4m3fn expert weights in tiles (csrc/experts_tiles.hip); the
    silu stage re-quantizes via the fused silu_mul_fp8 kernel so no extra passes
    appear."""
    n = _native()
    (T, H), K, (E, _, I) = xq.data.shape, ids.shape[1], w2q.shape
    if T == 0:
        return torch.empty(0, H, dtype=torch.bfloat16, device=xq.data.device)
    bm = _moe_tile(T, K, E, 64)
    order, expert, place = _moe_sort(ids, E, H, I, bm)
    P = order.shape[0]
    new = lambda m: torch.empty(P, m, dtype=torch.bfloat16,
                                device=xq.data.device)
    h, y = new(2 * I), new(H)
    n.experts_tiles(h, xq.data, w13q, xq.scale, w13s, order, expert, False, K,
                    bm)
    a = silu_mul_q(h)
    n.experts_tiles(y, a.data, w2q, a.scale, w2s, order, expert, False, 0, bm)
    return _moe_sum(Choices(y, place, weights.float().contiguous()))


def decode_inputs(stage: torch.Tensor, rows: int, cap: int, pages: int,
                  io: dict) -> None:
    """Put the staged values of `rows` rows (csrc/decode_inputs.hip) into the
    input tensors of a captured decode step.  GPU."""
    _native().decode_inputs(stage, rows, cap, pages, io["input_ids"],
                            io["positions"], io["slot_mapping"],
                            io["seq_lens"], io.get("state_slots"),
                            io["block_tables"])


def greedy_sample(logits: torch.Tensor) -> torch.Tensor:
    if logits.is_cuda:
        out = torch.empty(logits.shape[0], dtype=torch.long,
                          device=logits.device)
        _native().greedy_sample(out, logits)
        return out
    return logits.float().argmax(-1)


def sample(logits: torch.Tensor, temperature: torch.Tensor,
           top_p: torch.Tensor, top_k: torch.Tensor,
           uniform: torch.Tensor) -> torch.Tensor:
    """Batch sampling: temperature (0: the largest logit), top-k, top-p and an
    inverse-CDF draw over the tokens in order of their ids, in one kernel or, of
    few rows, in two (csrc/sampling.hip)."""
    if not logits.is_cuda:
        return torch_ref.sample(logits, temperature, top_p, top_k, uniform)
    rows, vocab = logits.shape
    if top_k.dtype != torch.int32:
        top_k = top_k.clamp(0, vocab)
    # an option of one element is that of every row
    option = lambda t, kind: t.to(logits.device, kind).expand(rows) \
        .contiguous()
    temperature, top_p = (option(t, torch.float32)
                          for t in (temperature, top_p))
    top_k = option(top_k, torch.int32)
    if vocab >= 1 << 23:        # weights of up to 2^40 add up to 63 bits
        return torch_ref.sample(logits, temperature, top_p, top_k, uniform)
    if logits.dtype not in (torch.bfloat16, torch.float32):
        logits = logits.float()
    out = torch.empty(rows, dtype=torch.long, device=logits.device)
    _native().sample(out, logits.contiguous(), temperature, top_p, top_k,
                     uniform.to(logits.device, torch.float32).contiguous())
    return out
