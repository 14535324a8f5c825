"""ModelRunner: device-side execution of scheduled batches.

Decode steps are captured into hipGraphs per batch-size bucket (torch's CUDA
graph API is hipGraph on ROCm).  The capture includes the whole transformer
forward — custom CDNA4 kernels, library GEMMs and (at TP>1) the RCCL
all-reduces — so steady-state decode replays with one graph launch instead
of ~1k kernel launches (MI355X boundary cost ≈1.2-1.9 us each, see
/opt/skills/guides/MI355X_MICROARCH.md 'boundary').
"""

from __future__ import annotations

import logging
import os
from typing import Dict, List, Optional

import torch

from hyperspot import ops
from hyperspot.models import build_model
from hyperspot.models.llama import (ABSORB_TOKENS, SPAN_TOKENS, ForwardMeta,
                                    LatentSpan, prefill_tiles)

from .config import EngineConfig
from .kv_cache import (BlockManager, allocate_caches,
                       compute_num_gpu_blocks)
from .request import Request
from .scheduler import ScheduledBatch

log = logging.getLogger(__name__)

_TUNABLEOP_LOADED = False


def _load_tunableop_results() -> None:
    """Load committed hipBLASLt algo selections (profiles/tunableop_gfx950.csv).

    The default hipBLASLt heuristic picks ~1.5-3x-off-roofline kernels for
    the skinny decode GEMMs (M=64..256); offline tuning (tools/tune_gemms.py
    on an MI355X) selects per-shape algorithms which TunableOp then replays.
    No tuning happens at serve time — results are read-only.
    """
    global _TUNABLEOP_LOADED
    if _TUNABLEOP_LOADED:
        return
    _TUNABLEOP_LOADED = True
    path = os.path.join(os.path.dirname(os.path.dirname(
        os.path.dirname(os.path.abspath(__file__)))),
        "profiles", "tunableop_gfx950.csv")
    if not os.path.exists(path):
        return
    try:
        t = torch.cuda.tunable
        t.enable(True)
        t.tuning_enable(False)   # replay only; never tune in the hot path
        t.record_untuned_enable(False)
        t.read_file(path)
        log.info("TunableOp: loaded %s", path)
    except Exception as e:  # pragma: no cover
        log.warning("TunableOp load failed: %s", e)


# Prompts of between a half and three quarters of a captured size would be mostly
# padded, which takes its share of the products, and in layers of experts reads the
# weights of those that it chooses.  So five and six eighths of a size are captured
# as well.  us, padded to the size and to the step: 540 tokens, 8 wide layers 3814 ->
# 2967, 8 narrow ones 1587 -> 1286, 4 of Mixtral 8x7B 4791 -> 3309; 270 2195 -> 1945,
# 995 -> 886, 4153 -> 2534; 1500 6394 -> 5306, 2467 -> 2132, 7350 -> 5777.  Seven
# eighths gain less, or lose (1792 rows of wide layers 6437 6774); steps of decoded
# rows, whose sizes lie closer, stay as they are (150 rows 1764 1813, 130 869 860).
# Each costs a capture at startup: of Llama-3-8B 13 prompt graphs take 0.34 s where 5
# took 0.16, and all graphs 1068 MB in place of 706.
#
# Steps are whole tiles of 32 rows: eighths of any size are not, and latent attention
# takes 8 rows at a time.
def _between(size: int) -> List[int]:
    """The steps below a captured size, from 256 on."""
    return [-(-size * k // 256) * 32 for k in (5, 6)] if size >= 256 else []


def _with_between(sizes) -> List[int]:
    """The sizes, and the steps between those from 256 on."""
    out, before = [], 0
    for s in sizes:
        out += [t for t in _between(s) if t > before]
        out.append(s)
        before = s
    return out


def _nearest(n: int, size: int, captured) -> int:
    """`size`, or the smallest captured step below it that holds n: without
    capture_all_graphs there is none, for a step that has to capture first takes the
    sizes themselves."""
    for t in _between(size):
        if n <= t and t in captured:
            return t
    return size


class ModelRunner:
    def __init__(self, config: EngineConfig, device: Optional[str] = None):
        self.config = config
        self.spec = config.spec()
        if config.max_model_len > self.spec.max_position:
            # the rope table is sized for max_position; admitting longer
            # prompts crashed the stepping thread with an index OOB
            log.warning("max_model_len %d clamped to the model's "
                        "max_position %d", config.max_model_len,
                        self.spec.max_position)
            config.max_model_len = self.spec.max_position
        self.device = torch.device(
            device if device is not None
            else ("cuda" if torch.cuda.is_available() else "cpu"))
        hybrid = self.spec.is_hybrid
        if config.dtype not in ("bfloat16", "float32"):
            raise ValueError(f"unknown dtype {config.dtype!r}")
        if config.dtype == "float32" and self.device.type == "cuda":
            if not hybrid:
                raise ValueError(f"{config.model}: this family's GPU kernels "
                                 "are bfloat16 only")
            torch.backends.cuda.matmul.allow_tf32 = False
            torch.set_float32_matmul_precision("highest")
        if hybrid and (config.quant or config.kv_dtype != "bfloat16"):
            raise ValueError(f"{config.model}: fp8 weights and fp8 KV pages "
                             "are not available for this design")
        if self.spec.has_state and config.enable_prefix_caching:
            log.warning("prefix caching is off: %s keeps recurrent state, "
                        "which shared pages do not restore", config.model)
            config.enable_prefix_caching = False
        self.dtype = torch.bfloat16 if self.device.type == "cuda" \
            and config.dtype == "bfloat16" else torch.float32
        torch.manual_seed(config.seed)
        if self.device.type == "cuda":
            _load_tunableop_results()
        from hyperspot.parallel.layers import set_init_device, set_quant_mode
        set_init_device(self.device)
        set_quant_mode(config.quant)
        self.model = build_model(self.spec, dtype=self.dtype).to(self.device)
        self.model.eval()
        if os.path.isdir(config.model):
            from .checkpoint import load_pretrained
            load_pretrained(self.model, config.model)
        # a sequence's table row is also its recurrent-state slot
        rows = config.max_num_seqs if self.spec.has_state \
            else max(config.max_num_seqs * 2, 64)
        self.num_blocks = compute_num_gpu_blocks(
            self.spec, config, self.device,
            num_slots=rows if self.spec.has_state else 0)
        assert config.kv_dtype in ("bfloat16", "fp8"), config.kv_dtype
        kv_dt = torch.float8_e4m3fn if config.kv_dtype == "fp8" \
            else self.dtype
        self.kv_caches = allocate_caches(self.spec, config, self.num_blocks,
                                         rows, kv_dt, self.device)
        self.max_blocks_per_seq = (config.max_model_len + config.block_size - 1) \
            // config.block_size
        self.block_manager = BlockManager(
            self.num_blocks, config.block_size,
            capacity=rows,
            max_blocks_per_seq=self.max_blocks_per_seq,
            enable_prefix_caching=config.enable_prefix_caching)
        self._gen = torch.Generator().manual_seed(config.seed)
        # pinned staging for the decode hot path (vectorized input prep)
        pin = self.device.type == "cuda"
        cap = self.block_manager.capacity
        # [id | position | slot | tokens | state row] of cap int64 each, then
        # the page ids as int32
        self._stage = torch.empty(
            5 * cap + (cap * self.max_blocks_per_seq + 1) // 2,
            dtype=torch.long, pin_memory=pin)
        self._stage_dev = torch.empty_like(self._stage, device=self.device) \
            if pin else self._stage
        self._st_event = torch.cuda.Event() if pin else None
        self._st_stream = None          # of the last decode step
        # guided-decoding logit-mask rows keyed by machine state
        self._guided_mask_cache: Dict[tuple, torch.Tensor] = {}
        self._graphs: Dict[int, torch.cuda.CUDAGraph] = {}
        self._graph_io: Dict[int, dict] = {}
        self._pgraphs: Dict[int, torch.cuda.CUDAGraph] = {}
        self._pgraph_io: Dict[int, dict] = {}
        self._graph_pool = None

    # ---------------- input preparation ----------------

    def _to_device(self, *parts) -> List[torch.Tensor]:
        """numpy arrays (int64 or int32) on the device, by one copy that the
        host does not wait for."""
        import numpy as np
        size = [-(-p.nbytes // 8) for p in parts]
        cuda = self.device.type == "cuda"
        host = torch.empty(sum(size), dtype=torch.long, pin_memory=cuda)
        at, flat = 0, host.numpy()
        for p, n in zip(parts, size):
            flat[at:at + n].view(p.dtype)[:p.size] = p.reshape(-1)
            at += n
        dev = host.to(self.device, non_blocking=cuda)
        out, at = [], 0
        for p, n in zip(parts, size):
            t = dev[at:at + n]
            if p.dtype == np.int32:
                t = t.view(torch.int32)[:p.size]
            out.append(t.view(p.shape))
            at += n
        return out

    def _prefill_inputs(self, batch: ScheduledBatch):
        import numpy as np
        bm = self.block_manager
        bs = bm.block_size
        rows = [bm.row_of[r.request_id] for r in batch.requests]
        begin = [r.chunk_start for r in batch.requests]
        lens = [r.chunk_len or r.num_prompt_tokens for r in batch.requests]
        starts = np.cumsum([0] + lens, dtype=np.int32)
        ids = np.concatenate([np.asarray(r.tokens(b, n), dtype=np.int64)
                              for r, b, n in zip(batch.requests, begin,
                                                 lens)])
        seq = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
        pos = np.arange(starts[-1], dtype=np.int64) \
            + np.repeat(np.asarray(begin) - starts[:-1], lens)
        slots = bm.tables_np[np.repeat(rows, lens), pos // bs] \
            .astype(np.int64) * bs + pos % bs
        nt = bm.ntables_np[rows]
        table = bm.tables_np[rows, :int(nt.max())]
        table = np.where(np.arange(table.shape[1]) < nt[:, None], table, 0) \
            .astype(np.int32)
        (input_ids, positions, slots, last, seq_start, seq, ctx,
         table) = self._to_device(
            ids, pos, slots, (starts[1:] - 1).astype(np.int64), starts, seq,
            (pos + 1).astype(np.int32), table)
        meta = ForwardMeta(
            mode="prefill", positions=positions, slot_mapping=slots,
            seq_start=seq_start, max_seqlen=max(lens), min_seqlen=min(lens),
            # a continuation chunk attends over the cache
            fresh_prefill=not any(begin),
            row_seq=seq, ctx_lens=ctx, block_tables=table,
            logits_indices=last)
        if self.spec.is_hybrid:
            self._add_hybrid_meta(meta, rows, lens)
            if self.device.type == "cuda":
                meta.latent = {w: self._latent_span(w, rows, begin, lens)
                               for w in self.spec.latent_windows}
        return input_ids, meta

    def _add_hybrid_meta(self, meta: ForwardMeta, rows: List[int],
                        lens: List[int]) -> None:
        """State slots and tile list of a prefill step, one copy to the
        device: [slots | tile_start | tiles]."""
        tiles, tile_start = prefill_tiles(lens)
        flat = rows + tile_start + [x for t in tiles for x in t]
        dev = torch.tensor(flat, dtype=torch.int32, device=self.device)
        n = len(rows)
        meta.state_slots = dev[:n]
        meta.tile_start = dev[n:2 * n + 1]
        meta.tiles = dev[2 * n + 1:].view(-1, 2)

    def _latent_span(self, window: int, rows: List[int], begin: List[int],
                     lens: List[int]) -> LatentSpan:
        """Work lists of latent attention (see LatentSpan) for portions that
        begin at these positions."""
        import numpy as np
        bm = self.block_manager
        slots, start, first, short, n, row0 = [], [], [], [], 0, 0
        for row, b, m in zip(rows, begin, lens):
            start.append(n)
            first.append(max(0, b - window + 1))
            if m <= ABSORB_TOKENS:
                short += range(row0, row0 + m)
            else:
                p = np.arange(first[-1], b + m)
                s = bm.tables_np[row, p // bm.block_size].astype(np.int64) \
                    * bm.block_size + p % bm.block_size
                pad = -len(p) % 8
                slots += [s, np.full(pad, -1)] if pad else [s]
                n += len(p) + pad
            row0 += m
        tiles = [[i, a] for i, m in enumerate(lens) if m > ABSORB_TOKENS
                 for a in range(0, m, SPAN_TOKENS)]
        flat = start + first + [x for t in tiles for x in t] + short
        dev = torch.tensor(flat, dtype=torch.int32, device=self.device)
        k, t = len(rows), 2 * len(tiles)
        return LatentSpan(
            torch.from_numpy(np.concatenate(slots) if slots
                             else np.empty(0, np.int64)).to(self.device),
            dev[:k], dev[k:2 * k], dev[2 * k:2 * k + t].view(-1, 2),
            dev[2 * k + t:] if short else None)

    def _decode_inputs(self, batch: ScheduledBatch):
        """Vectorized decode-step prep: numpy state + pinned staging (the
        per-sequence Python loop cost more than the GPU step at batch 256),
        one copy to the device.  (staged values, rows, page ids a row)"""
        import numpy as np
        bm = self.block_manager
        reqs = batch.requests
        B = len(reqs)
        rows = np.fromiter((bm.row_of[r.request_id] for r in reqs),
                           dtype=np.int64, count=B)
        ids = np.fromiter((r.last_token_id for r in reqs),
                          dtype=np.int64, count=B)
        pos = bm.tokens_np[rows].copy()             # next position index
        slots = bm.append_slots_batch(rows)
        max_nt = int(bm.ntables_np[rows].max())
        bt = bm.tables_np[rows[:, None], np.arange(max_nt)[None, :]]
        if self._st_event is not None:
            # the last step's copy may still be reading the staging buffer: a
            # step need not end in a device synchronization
            self._st_event.synchronize()
            # nor run on this one's stream, which writes where it reads
            stream = torch.cuda.current_stream(self.device)
            if self._st_stream not in (None, stream):
                stream.wait_stream(self._st_stream)
            self._st_stream = stream
        cap = bm.capacity
        used = 5 * cap + (B * max_nt + 1) // 2
        st = self._stage.numpy()
        for i, x in enumerate((ids, pos, slots, pos + 1, rows)):
            st[i * cap:i * cap + B] = x
        st[5 * cap:].view(np.int32)[:B * max_nt] = bt.reshape(-1)
        d = self._stage_dev
        if self._st_event is not None:
            d[:used].copy_(self._stage[:used], non_blocking=True)
            self._st_event.record()
        return d, B, max_nt

    def _decode_meta(self, staged):
        """Tensors of an eager decode step from the staged values."""
        d, B, max_nt = staged
        cap = self.block_manager.capacity
        part = lambda i: d[i * cap:i * cap + B].clone()
        meta = ForwardMeta(
            mode="decode", positions=part(1), slot_mapping=part(2),
            block_tables=d[5 * cap:].view(torch.int32)[:B * max_nt]
            .clone().view(B, max_nt),
            seq_lens=part(3).to(torch.int32))
        if self.spec.is_hybrid:
            meta.state_slots = part(4).to(torch.int32)
        return part(0), meta

    # ---------------- execution ----------------

    @torch.inference_mode()
    def execute(self, batch: ScheduledBatch) -> torch.Tensor:
        """Run one step; returns sampled token ids [num_seqs] (cpu)."""
        return self._sample(self.forward(batch), batch.requests)

    @torch.inference_mode()
    def forward(self, batch: ScheduledBatch, want=None,
                trail: Optional[list] = None) -> torch.Tensor:
        """Run one step's forward; logits of every sequence's last token
        [num_seqs, vocab], or of the places `want` lists per sequence (places
        within its portion) in that order.  `trail` collects the residual
        stream after every layer (prefill steps, eager)."""
        if batch.mode == "decode" and trail is None:
            logits = self._decode_forward(self._decode_inputs(batch))
            if want is not None:
                logits = logits[[i for i, w in enumerate(want) for _ in w]]
            return logits
        if want is None and trail is None:
            logits = self._prefill_graph_forward(batch)
            if logits is not None:
                return logits
        input_ids, meta = self._prefill_inputs(batch)
        meta.residual_trail = trail
        if want is not None:
            starts = meta.seq_start.tolist()
            meta.logits_indices = torch.tensor(
                [a + p for a, w in zip(starts, want) for p in w],
                dtype=torch.long, device=self.device)
        return self.model(input_ids, meta, self.kv_caches)

    # ---- TTFT fast path: single-request whole-prompt prefill graphs ----

    def _prefill_bucket(self, n: int) -> Optional[int]:
        for s in self.config.prefill_graph_sizes:
            if s >= n and s <= self.config.max_num_batched_tokens:
                return s
        return None

    def _prefill_graph_forward(self, batch: ScheduledBatch):
        """Replay a padded single-sequence prefill graph (eager prefill
        costs ~350 kernel launches + the Python layer loop — several ms
        of the TTFT).  Pad tokens sit AFTER the real prompt, so causal
        attention keeps real rows exact; padded slots are -1 (no KV
        write) and the single logit row indexes the real last token."""
        if (self.device.type != "cuda" or self.config.enforce_eager
                or len(batch.requests) != 1):
            return None
        req = batch.requests[0]
        n = req.chunk_len or req.num_prompt_tokens
        if req.chunk_start != 0 or n != req.num_prompt_tokens:
            return None              # chunked / continued prompt
        T = self._prefill_bucket(n)
        if T is None:
            return None
        T = _nearest(n, T, self._pgraphs)
        if T not in self._pgraphs:
            self._capture_prefill(T)
        import numpy as np
        bm = self.block_manager
        row = bm.row_of[req.request_id]
        p = np.arange(n)
        io = self._pgraph_io[T]
        # one copy into the graph's inputs; pad tokens write no page
        host = torch.zeros(io["inputs"].numel(), dtype=torch.long,
                           pin_memory=True)
        at = host.numpy()
        at[:n] = req.prompt_token_ids[:n]
        at[T:T + n] = p
        at[2 * T:2 * T + n] = bm.tables_np[row, p // bm.block_size] \
            .astype(np.int64) * bm.block_size + p % bm.block_size
        at[2 * T + n:3 * T] = -1
        at[3 * T] = n - 1
        io["inputs"].copy_(host, non_blocking=True)
        if self.spec.is_hybrid:
            d = self.device
            # the recurrence must stop at the last real token
            io["seq_start"][1] = n
            io["state_slots"][0] = row
            io["block_tables"][0, :int(bm.ntables_np[row])] = torch.from_numpy(
                bm.tables_np[row, :int(bm.ntables_np[row])]).to(d)
        self._pgraphs[T].replay()
        return io["logits"]

    def _capture_prefill(self, T: int) -> None:
        d = self.device
        log.info("capturing prefill hipGraph for tokens=%d", T)
        inputs = torch.zeros(3 * T + 1, dtype=torch.long, device=d)
        inputs[2 * T:3 * T] = -1
        io = {
            "inputs": inputs,
            "input_ids": inputs[:T],
            "positions": inputs[T:2 * T],
            "slot_mapping": inputs[2 * T:3 * T],
            "lidx": inputs[3 * T:],
            "seq_start": torch.tensor([0, T], dtype=torch.int32, device=d),
        }
        meta = ForwardMeta(
            mode="prefill", positions=io["positions"],
            slot_mapping=io["slot_mapping"],
            seq_start=io["seq_start"],
            max_seqlen=T, fresh_prefill=True,
            logits_indices=io["lidx"], padded=True)
        if self.spec.is_hybrid:
            self._add_hybrid_meta(meta, [-1], [T])
            io["state_slots"] = meta.state_slots
            io["block_tables"] = torch.zeros(
                1, self.max_blocks_per_seq, dtype=torch.int32, device=d)
            meta.block_tables = io["block_tables"]
            meta.row_seq = torch.zeros(T, dtype=torch.int32, device=d)
            # a whole prompt: its tokens are the kv rows, one to one
            zero = torch.zeros(1, dtype=torch.int32, device=d)
            tiles = torch.tensor(prefill_tiles([T], SPAN_TOKENS)[0],
                                 dtype=torch.int32, device=d)
            meta.latent = {w: LatentSpan(io["slot_mapping"], zero, zero,
                                         tiles, None)
                           for w in self.spec.latent_windows}
        # the graph reads every tensor of meta at each replay: keep them all
        io["meta"] = meta
        for _ in range(2):
            self.model(io["input_ids"], meta, self.kv_caches)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, pool=self._graph_pool):
            io["logits"] = self.model(io["input_ids"], meta,
                                      self.kv_caches)
        if self._graph_pool is None:
            self._graph_pool = g.pool()
        self._pgraphs[T] = g
        self._pgraph_io[T] = io

    def _decode_forward(self, staged):
        stage, B, max_nt = staged
        bucket = self._bucket_for(B)
        if bucket is None or self.device.type != "cuda" \
                or self.config.enforce_eager:
            input_ids, meta = self._decode_meta(staged)
            return self.model(input_ids, meta, self.kv_caches)
        if bucket not in self._graphs:
            self._capture(bucket)
        io = self._graph_io[bucket]
        ops.decode_inputs(stage, B, self.block_manager.capacity, max_nt, io)
        self._graphs[bucket].replay()
        return io["logits"][:B]

    def _bucket_for(self, b: int) -> Optional[int]:
        for s in self.config.graph_batch_sizes:
            if s >= b:
                return s
        return None

    def _capture(self, bucket: int) -> None:
        d = self.device
        log.info("capturing decode hipGraph for batch=%d", bucket)
        io = {
            "input_ids": torch.zeros(bucket, dtype=torch.long, device=d),
            "positions": torch.zeros(bucket, dtype=torch.long, device=d),
            "slot_mapping": torch.full((bucket,), -1, dtype=torch.long, device=d),
            "block_tables": torch.zeros(bucket, self.max_blocks_per_seq,
                                        dtype=torch.int32, device=d),
            "seq_lens": torch.ones(bucket, dtype=torch.int32, device=d),
        }
        meta = ForwardMeta(mode="decode", positions=io["positions"],
                           slot_mapping=io["slot_mapping"],
                           block_tables=io["block_tables"],
                           seq_lens=io["seq_lens"], padded=True)
        if self.spec.is_hybrid:
            io["state_slots"] = torch.full((bucket,), -1, dtype=torch.int32,
                                           device=d)
            meta.state_slots = io["state_slots"]
        io["meta"] = meta            # the graph reads its tensors
        # warmup outside capture (allocator, hipBLASLt heuristics, RCCL)
        for _ in range(2):
            self.model(io["input_ids"], meta, self.kv_caches)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, pool=self._graph_pool):
            io["logits"] = self.model(io["input_ids"], meta, self.kv_caches)
        if self._graph_pool is None:
            self._graph_pool = g.pool()
        self._graphs[bucket] = g
        self._graph_io[bucket] = io

    @torch.inference_mode()
    def capture_all_graphs(self) -> None:
        # inference_mode matches the lazy in-step captures: every graph
        # io tensor is an inference tensor regardless of capture origin
        # (mixing modes trips "inplace update to inference tensor")
        if self.device.type != "cuda" or self.config.enforce_eager:
            return
        for b in self.config.graph_batch_sizes:
            if b <= self.config.max_num_seqs and b not in self._graphs:
                self._capture(b)
        for t in _with_between(s for s in self.config.prefill_graph_sizes
                               if s <= self.config.max_num_batched_tokens):
            if t <= self.config.max_model_len and t not in self._pgraphs:
                self._capture_prefill(t)

    # ---------------- embeddings ----------------

    @torch.inference_mode()
    def embed(self, prompts: List[List[int]]) -> torch.Tensor:
        """Mean-pooled final hidden state per prompt -> [N, hidden] fp32.

        Runs outside the scheduler on temporary KV pages (freed at the end);
        serves the llm-gateway /embeddings contract."""
        free = self.block_manager.num_free_rows
        if free == 0:
            raise RuntimeError("no free sequence slots for embeddings")
        return torch.cat([self._embed_group(prompts[i:i + free])
                          for i in range(0, len(prompts), free)])

    def _embed_group(self, prompts: List[List[int]]) -> torch.Tensor:
        from .request import Request
        from .config import SamplingParams
        bm = self.block_manager
        fake = []
        try:
            for i, p in enumerate(prompts):
                rid = f"__embed_{i}"
                bm.allocate(rid, len(p))
                fake.append(Request(request_id=rid, prompt_token_ids=list(p),
                                    sampling=SamplingParams()))
            batch = ScheduledBatch(mode="prefill", requests=fake,
                                   num_tokens=sum(len(p) for p in prompts))
            input_ids, meta = self._prefill_inputs(batch)
            meta.return_hidden = True
            hidden = self.model(input_ids, meta, self.kv_caches).float()
            out = torch.empty(len(prompts), hidden.shape[-1],
                              dtype=torch.float32, device=hidden.device)
            ss = meta.seq_start
            for i in range(len(prompts)):
                out[i] = hidden[int(ss[i]):int(ss[i + 1])].mean(0)
        finally:
            for i in range(len(prompts)):
                bm.free(f"__embed_{i}")
        return out.cpu()

    def swap_weights(self, checkpoint_path: str) -> float:
        from .checkpoint import load_checkpoint_into
        return load_checkpoint_into(self.model, checkpoint_path)

    # ---------------- sampling ----------------

    def _apply_guided(self, logits: torch.Tensor,
                      requests: List[Request]) -> None:
        """Structured-output mask (SamplingParams.response_format="json"):
        only grammar-legal next BYTES (byte tokenizer: id = byte + 4)
        keep their logits; EOS opens up once the JSON value is closed.
        In-place on the [B, vocab] logits; no-op without guided seqs."""
        gis = [i for i, r in enumerate(requests)
               if r.sampling.response_format in ("json", "tool_call")
               or r.sampling.response_schema is not None]
        if not gis:
            return
        from .guided import (JsonByteMachine, SchemaMachine,
                             ToolCallMachine)
        NB = 4 + 256                       # specials + byte ids
        neg = float("-inf")
        rows: List[torch.Tensor] = []
        cache = self._guided_mask_cache
        for k, i in enumerate(gis):
            r = requests[i]
            m = getattr(r, "_guided", None)
            if m is None or m.consumed > len(r.output_token_ids):
                if r.sampling.response_format == "tool_call":
                    m = ToolCallMachine(tuple(r.sampling.tool_names))
                elif r.sampling.response_schema is not None:
                    try:
                        # untrusted schema: any compile failure degrades
                        # to plain JSON-grammar enforcement
                        m = SchemaMachine(r.sampling.response_schema)
                    except Exception:
                        m = JsonByteMachine()
                else:
                    m = JsonByteMachine()
                r._guided = m
            for t in r.output_token_ids[m.consumed:]:
                m.feed_token(t)
            # cache mask rows by machine state (mask_key): avoids a
            # ~230-iteration Python loop per guided sequence per step
            key = m.mask_key() if hasattr(m, "mask_key") else None
            row = cache.get(key) if key is not None else None
            if row is None:
                allow, eos_ok = m.allowed()
                row = torch.full((NB,), neg, dtype=torch.float32)
                for b in allow:
                    row[b + 4] = 0.0
                if eos_ok:
                    row[2] = 0.0           # ByteTokenizer EOS
                if key is not None:
                    cache[key] = row
            rows.append(row)
        small = torch.stack(rows)
        d = logits.device
        gidx = torch.tensor(gis, device=d)
        logits[gidx, NB:] = neg
        logits[gidx, :NB] += small.to(device=d, dtype=logits.dtype)

    def _sample(self, logits: torch.Tensor, requests: List[Request]) -> torch.Tensor:
        B = logits.shape[0]
        self._apply_guided(logits, requests)
        temps = torch.tensor([r.sampling.temperature for r in requests],
                             dtype=torch.float32)
        if bool((temps == 0).all()):
            return ops.greedy_sample(logits).cpu()
        top_p = torch.tensor([r.sampling.top_p for r in requests],
                             dtype=torch.float32)
        top_k = torch.tensor([r.sampling.top_k for r in requests],
                             dtype=torch.int32)
        if any(r.sampling.seed is not None for r in requests):
            # per-request reproducible draws (SamplingParams.seed)
            us = []
            for r in requests:
                if r.sampling.seed is not None:
                    g = getattr(r, "_seed_gen", None)
                    if g is None:
                        g = torch.Generator().manual_seed(r.sampling.seed)
                        r._seed_gen = g
                    us.append(torch.rand(1, generator=g))
                else:
                    us.append(torch.rand(1, generator=self._gen))
            uniform = torch.cat(us)
        else:
            uniform = torch.rand(B, generator=self._gen)
        d = logits.device
        return ops.sample(logits, temps.to(d), top_p.to(d), top_k.to(d),
                          uniform.to(d)).cpu()
