"""Op dispatch layer.

On GPU (ROCm) every hot op runs a hand-written CDNA4 HIP kernel from the
in-tree extension ``hyperspot._C`` (csrc/, built for gfx950 only).  On CPU the
pure-PyTorch references in :mod:`hyperspot.ops.torch_ref` run instead (CI has
no GPU).  There is no CUDA path, no Triton, no multi-backend dispatch — a CUDA
device without the extension is a hard error, never a silent eager fallback.
"""

from __future__ import annotations

from typing import NamedTuple

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


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().rmsnorm(out, x, weight, eps)
        return out
    return torch_ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor,
                      weight: torch.Tensor, eps: float):
    """residual += x (in place); x_out = rmsnorm(residual) (in place on x)."""
    if x.is_cuda:
        _native().fused_add_rmsnorm(x, residual, weight, eps)
        return x, residual
    out, res = torch_ref.fused_add_rmsnorm(x, residual, weight, eps)
    return out, res


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


def paged_attn_decode(q: torch.Tensor, k_cache: torch.Tensor,
                      v_cache: torch.Tensor, block_tables: torch.Tensor,
                      seq_lens: torch.Tensor, scale: float) -> torch.Tensor:
    if q.is_cuda:
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        kvh = k_cache.shape[1]
        split = _attn_split(q.shape[0], kvh) if q.shape[-1] == 128 else 1
        ws = None
        if split > 1:
            ws = torch.empty(q.shape[0] * kvh * split
                             * (q.shape[1] // kvh) * 130,
                             dtype=torch.float32, device=q.device)
        _native().paged_attn(out, q, k_cache, v_cache, block_tables,
                             seq_lens, None, scale, ws, split)
        return out
    return torch_ref.paged_attn_decode(q, k_cache, v_cache, block_tables,
                                       seq_lens, scale)


# Portions of at least this many rows attend on the matrix cores.  A tile of
# 32 rows costs what it costs for one row, and has no other workgroups to share
# its keys with; the row-by-row kernel reads the keys once per row, but spreads
# them over more workgroups.  16 rows after 16000 tokens: 387 us against 473;
# after 1000: 29 us against 35; 8 kv heads of 4 query heads.
PORTION_ROWS = 16


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
                and q.shape[1] // k_cache.shape[1] in (1, 2, 4, 8):
            _native().attn_portions(
                out, q, k_cache, v_cache, meta.block_tables, meta.ctx_lens,
                meta.row_seq, meta.seq_start, PORTION_ROWS,
                getattr(meta, "min_seqlen", 0) < PORTION_ROWS, scale)
        else:
            # row by row: odd head dims
            _native().paged_attn(out, q, k_cache, v_cache,
                                 meta.block_tables, meta.ctx_lens,
                                 meta.row_seq, scale, None, 1)
        return out
    if getattr(meta, "fresh_prefill", True):
        return torch_ref.prefill_attn(q, k, v, meta.seq_start, scale)
    return torch_ref.prefill_attn_paged(q, k_cache, v_cache,
                                        meta.block_tables, meta.ctx_lens,
                                        meta.row_seq, scale)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    if gate_up.is_cuda:
        i = gate_up.shape[-1] // 2
        out = torch.empty(*gate_up.shape[:-1], i, dtype=gate_up.dtype,
                          device=gate_up.device)
        _native().silu_mul(out, gate_up)
        return out
    return torch_ref.silu_mul(gate_up)


def _rows_gemm(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether csrc/gemm_rows.hip takes x w^T: few rows, and a weight whose
    tiles of 16 rows divide evenly over the 256 compute units; the library is
    as fast or faster elsewhere (us, library and kernel, one row: 6144 x 4096
    14.4 14.8, 4096 x 14336 26.9 28.0, 2048 x 7168 13.2 13.2)."""
    if not (x.is_cuda and x.dtype == w.dtype == torch.bfloat16
            and x.dim() == 2 and w.dim() == 2 and 1 <= x.shape[0] <= 64):
        return False
    (M, K), N = x.shape, w.shape[0]
    tiles = (N + 15) // 16
    if K > 4096 or K % 8 or N % 4 or N * K < (1 << 20) \
            or -(-tiles // 256) * 256 > 1.2 * tiles and tiles > 256:
        return False
    return _native().gemm_rows_fits(M, K) and all(
        t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0
        for t in (x, w))


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x w^T for w [N, K]."""
    if _rows_gemm(x, w):
        out = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype,
                          device=x.device)
        _native().gemm_rows(out, x, w)
        return out
    return x @ w.t()


class QTensor(NamedTuple):
    """Per-token-scaled fp8 activation: data e4m3fn [T,K], scale fp32 [T].

    Produced on GPU by the fused quant kernels (csrc/quant.hip) so fp8
    GEMM inputs never take an extra elementwise pass; consumed by the TP
    linear layers via torch._scaled_mm (hipBLASLt fp8 MFMA)."""

    data: torch.Tensor
    scale: torch.Tensor


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
    assert x.is_cuda
    T, K = x.shape
    out = torch.empty(T, K, dtype=torch.float8_e4m3fn, device=x.device)
    scales = torch.empty(T, dtype=torch.float32, device=x.device)
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
    """Split-K degree + fp32 workspace for a grouped GEMM launch.

    The w2 GEMM at Mixtral decode shapes has ~288 blocks for 256 CUs —
    its ragged second wave idles most of the chip; splitting K into up
    to 8 segments (each must keep >= 3 k-chunks for the LDS ring and
    divide the chunk count) multiplies the block count back above ~4
    per CU.  Shapes-only decision: hipGraph-capture-safe.
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


def moe_router(x, router: torch.Tensor, top: int):
    """(weights [T, top] float, expert ids [T, top] int32) of the rows of x, a
    bf16 tensor or a QTensor: the softmax over the chosen.  GPU."""
    data, scale = x if isinstance(x, QTensor) else (x, None)
    T = data.shape[0]
    weight = torch.empty(T, top, dtype=torch.float32, device=data.device)
    ids = torch.empty(T, top, dtype=torch.int32, device=data.device)
    _native().experts_router(weight, ids, data, scale, router, top)
    return weight, ids


# Rows per expert up to which tiles of 16 to 64 rows beside the streamed weights
# are faster than the 256-row tiles, in us on an MI355X:
#   experts of 14336 x 4096  1 row 274 : 463, 48 rows 788 : 831, 64 1049 : 846
#   32 of 1024 x 2048        1 row  54 : 157, 64 rows 180 : 277, 128 269 : 305
#   16 of 2048 x 4096        1 row 132 : 273, 64 rows 335 : 378,  96 397 : 391
# The large tiles are late where they leave compute units without one.
MOE_ROWS = 48
MOE_ROWS_FEW = 95


def _moe_rows(T: int, K: int, E: int, H: int, I: int) -> bool:
    most = MOE_ROWS_FEW if E * (2 * I // 128) < 1024 else MOE_ROWS
    return T * K <= most * E and H % 128 == 0 and I % 128 == 0 and E <= 64


def _moe_ffn_rows(x, w13, w2, weights, ids):
    n = _native()
    (T, H), K, (E, _, I) = x.shape, ids.shape[1], w2.shape
    pairs, mean = T * K, T * K / E
    bm = 16 if mean <= 8 else 32 if mean <= 16 else 64
    tiles = min(pairs, (pairs + E * (bm - 1)) // bm)
    i32 = lambda m: torch.empty(m, dtype=torch.int32, device=x.device)
    order, expert, place = i32(tiles * bm), i32(tiles), i32(pairs)
    n.experts_sort(order, expert, place, ids.reshape(-1).to(torch.int32), E,
                   bm)
    h = torch.empty(tiles * bm, I, dtype=x.dtype, device=x.device)
    y = torch.empty(tiles * bm, H, dtype=x.dtype, device=x.device)
    n.experts_up(h, x, w13, None, order, expert, K, None, bm)
    n.experts_down(y, h, w2, None, order, expert, bm)
    out = torch.empty(T, H, dtype=x.dtype, device=x.device)
    n.experts_sum(out, y, place.view(T, K), weights.float().contiguous(),
                  None, None, None, None, 0.0)
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
    T, H = x.shape
    K = ids.shape[1]
    E = w13.shape[0]
    TK = T * K
    if x.is_contiguous() and _moe_rows(T, K, E, H, w2.shape[2]):
        return _moe_ffn_rows(x, w13, w2, weights, ids)
    ntiles = (TK + E * (MOE_BM - 1) + MOE_BM - 1) // MOE_BM
    P = ntiles * MOE_BM
    dev = x.device
    flat = ids.reshape(-1).to(torch.int32)
    sorted_ids = torch.empty(P, dtype=torch.int32, device=dev)
    tile_expert = torch.empty(ntiles, dtype=torch.int32, device=dev)
    inv_pos = torch.empty(TK, dtype=torch.int32, device=dev)
    n = _native()
    n.moe_align(sorted_ids, tile_expert, inv_pos, flat, E)
    I2 = w13.shape[1]
    h1 = torch.empty(P, I2, dtype=torch.bfloat16, device=dev)
    s1, ws1 = _moe_splitk(ntiles * (I2 // 128), H // 64, P * I2, dev)
    n.moe_gemm(h1, x, w13, sorted_ids, tile_expert, K, s1, ws1)
    a = silu_mul(h1)
    y = torch.empty(P, H, dtype=torch.bfloat16, device=dev)
    I = w2.shape[2]
    s2, ws2 = _moe_splitk(ntiles * (H // 128), I // 64, P * H, dev)
    n.moe_gemm(y, a, w2, sorted_ids, tile_expert, 0, s2, ws2)
    out = torch.empty(T, H, dtype=torch.bfloat16, device=dev)
    n.moe_combine(out, y, weights.float().contiguous(), inv_pos, K)
    return out


def moe_ffn_fp8(xq: "QTensor", w13q: torch.Tensor, w13s: torch.Tensor,
                w2q: torch.Tensor, w2s: torch.Tensor,
                weights: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
    """fp8 grouped expert FFN: e4m3fn activations (QTensor from the fused
    norm producer) x e4m3fn expert weights through
    v_mfma_f32_32x32x16_fp8_fp8; the silu stage re-quantizes via the fused
    silu_mul_fp8 kernel so no extra passes appear.  ~2x the bf16 MoE
    weight bandwidth (the binding constraint, profiles/r01)."""
    T, H = xq.data.shape
    K = ids.shape[1]
    E = w13q.shape[0]
    TK = T * K
    ntiles = (TK + E * (MOE_BM - 1) + MOE_BM - 1) // MOE_BM
    P = ntiles * MOE_BM
    dev = xq.data.device
    flat = ids.reshape(-1).to(torch.int32)
    sorted_ids = torch.empty(P, dtype=torch.int32, device=dev)
    tile_expert = torch.empty(ntiles, dtype=torch.int32, device=dev)
    inv_pos = torch.empty(TK, dtype=torch.int32, device=dev)
    n = _native()
    n.moe_align(sorted_ids, tile_expert, inv_pos, flat, E)
    I2 = w13q.shape[1]
    h1 = torch.empty(P, I2, dtype=torch.bfloat16, device=dev)
    s1, ws1 = _moe_splitk(ntiles * (I2 // 128), H // 128, P * I2, dev)
    n.moe_gemm_fp8(h1, xq.data, xq.scale, w13q, w13s, sorted_ids,
                   tile_expert, K, s1, ws1)
    a = silu_mul_q(h1)
    y = torch.empty(P, H, dtype=torch.bfloat16, device=dev)
    I = w2q.shape[2]
    s2, ws2 = _moe_splitk(ntiles * (H // 128), I // 128, P * H, dev)
    n.moe_gemm_fp8(y, a.data, a.scale, w2q, w2s, sorted_ids, tile_expert,
                   0, s2, ws2)
    out = torch.empty(T, H, dtype=torch.bfloat16, device=dev)
    n.moe_combine(out, y, weights.float().contiguous(), inv_pos, K)
    return out


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
    inverse-CDF draw over the tokens in order of their ids, in one kernel."""
    if not logits.is_cuda:
        return torch_ref.sample(logits, temperature, top_p, top_k, uniform)
    if logits.dtype not in (torch.bfloat16, torch.float32):
        logits = logits.float()
    out = torch.empty(logits.shape[0], dtype=torch.long, device=logits.device)
    f32 = lambda t: t.to(logits.device, torch.float32).contiguous()
    _native().sample(out, logits.contiguous(), f32(temperature), f32(top_p),
                     top_k.to(logits.device, torch.int32).contiguous(),
                     f32(uniform))
    return out
