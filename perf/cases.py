"""The work that serving has the engine do, as cases that can be timed.

Decoder stacks with the layers of the dense and the expert family are run
through the scheduler, the cache manager and the model runner, as the worker
runs them: decode steps at small, ordinary and large batches and contexts,
whole prompts, packs of prompts and prompts that are longer than a step, in
bfloat16 and with 8-bit weights and pages; and the draw of the next tokens.

The stacks are those that `bench.py --compare` measures (the dense one has the
layers of Llama-3-8B), and Mixtral 8x7B with fewer layers.
"""

import math
import random

import numpy as np
import torch

from hyperspot import ops
from hyperspot.engine import EngineConfig, LLMEngine, ModelSpec, SamplingParams
from hyperspot.engine.request import Request
from hyperspot.engine.scheduler import ScheduledBatch

BLOCK = EngineConfig.block_size
BUDGET = EngineConfig.max_num_batched_tokens    # tokens of a prefill step
MAX_LEN = 16384
DECODE_TOKENS = 256 * 1024                      # cached tokens of a case

# name: width, layers, heads, kv heads, feed-forward, vocabulary, experts,
# choices, rotary base
STACKS = {
    "llama-w2048": (2048, 8, 16, 4, 7168, 32768, 0, 0, 500000.0),
    "llama-w4096": (4096, 8, 32, 8, 14336, 32768, 0, 0, 500000.0),
    "mixtral-w2048": (2048, 8, 16, 4, 1024, 32768, 32, 4, 500000.0),
    "mixtral-8x7b-l4": (4096, 4, 32, 8, 14336, 32000, 8, 2, 1000000.0),
}


def _spec(name, layers=0):
    w, n, h, kv, ff, vocab, experts, choices, theta = STACKS[name]
    return ModelSpec(name, w, layers or n, h, kv, 128, ff, vocab,
                     rope_theta=theta, max_position=MAX_LEN,
                     num_experts=experts, num_experts_per_tok=choices)


class _Config(EngineConfig):
    def spec(self):
        return self.stack


def listed():
    def decode(name, stack, batch, context, fp8=False):
        return {"name": name, "what": "decode", "stack": stack,
                "batch": batch, "context": context, "fp8": fp8}

    def prefill(name, stack, prompts, length, fp8=False):
        return {"name": name, "what": "prefill", "stack": stack,
                "prompts": prompts, "length": length, "fp8": fp8}

    return [
        # one user's chat: the latency of a token
        decode("decode 1", "llama-w4096", 1, 1000),
        # few long conversations
        decode("decode 8 long", "llama-w4096", 8, 8000),
        # a lightly used server, a smaller model
        decode("decode 32", "llama-w2048", 32, 1000),
        # a full server: the largest decode step
        decode("decode 256", "llama-w4096", 256, 1000),
        # the same server with 8-bit weights and pages
        decode("decode 64 fp8", "llama-w4096", 64, 1000, fp8=True),
        # experts: a few users, and a full server
        decode("experts decode 4", "mixtral-w2048", 4, 1000),
        decode("experts decode 192", "mixtral-8x7b-l4", 192, 500),
        # time to the first token of one prompt
        prefill("prompt 512", "llama-w4096", 1, 512),
        # waiting prompts packed into steps: the budget cuts one of them
        prefill("prompts 16", "llama-w4096", 16, 1000),
        # a document: longer than a step
        prefill("prompt 16000", "llama-w4096", 1, 16000),
        prefill("experts prompts 4", "mixtral-8x7b-l4", 4, 500),
        # the next token of every sequence, with the options users set
        {"name": "sample 64", "what": "sample", "batch": 64,
         "vocab": 128256},
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "experts decode", "prefill",
                       "prefill", "experts prefill", "sample"])
    if kind == "sample":
        return {"what": "sample", "batch": _spread(rng, 1, 256),
                "vocab": rng.choice([32000, 32768, 50257, 128256])}
    dense = not kind.startswith("experts")
    stack = rng.choice([n for n, s in STACKS.items() if dense == (s[6] == 0)])
    case = {"what": kind.split()[-1], "stack": stack,
            "fp8": rng.random() < 0.2}
    if case["what"] == "decode":
        case["batch"] = _spread(rng, 1, 256)
        case["context"] = min(_spread(rng, 64, 12000),
                              DECODE_TOKENS // case["batch"])
    else:
        case["prompts"] = _spread(rng, 1, 24)
        case["length"] = min(_spread(rng, 32, 12000),
                             12000 // case["prompts"])
    return case


# ---------------------------------------------------------------- inputs

def _lengths(case):
    """Ragged lengths around the mean, none of which ends a page when
    decoding; the length itself for a single sequence."""
    n = case.get("batch") or case["prompts"]
    mean = case.get("context") or case["length"]
    if n == 1:
        out = [mean]
    else:
        rng = random.Random(mean * 1009 + n)
        out = [max(1, int(mean * rng.uniform(0.5, 1.5))) for _ in range(n)]
        out = [min(m, MAX_LEN - BLOCK) for m in out]
    if case["what"] == "decode":
        out = [m + (m % BLOCK == 0) for m in out]
    return out


def _like_trained(model, spec, gen, dev):
    """Two properties of trained weights that random ones lack.  A layer
    changes the residual stream by less than the stream is, so that rounding
    does not grow from layer to layer; and tokens choose experts decisively:
    an embedding lies along its experts' directions, which every layer's
    router reads in an order of its own."""
    e, w = spec.num_experts, spec.hidden_size
    if not e:
        model.embed.data.normal_(0.0, 4.0, generator=gen)
        return
    basis, _ = torch.linalg.qr(torch.randn(w, e, generator=gen, device=dev))
    basis = basis.t() * w ** 0.5                         # rows of norm sqrt(w)
    rank = torch.rand(spec.vocab_size, e, generator=gen, device=dev)
    order = rank.argsort(-1)[:, :spec.num_experts_per_tok]
    shares = torch.linspace(1.0, 0.7, spec.num_experts_per_tok, device=dev)
    emb = torch.randn(spec.vocab_size, w, generator=gen, device=dev)
    for c in range(spec.num_experts_per_tok):
        emb += 6 * shares[c] * basis[order[:, c]]
    model.embed.data.copy_(emb)
    for layer in model.layers:
        perm = torch.randperm(e, generator=gen, device=dev)
        layer.mlp.moe.router.data.copy_(basis[perm] * (0.1 / w ** 0.5))


def _engine(case, lengths):
    # fewer layers with 8 bits: what rounding to 8 bits does to a value that
    # is changed a little grows from layer to layer
    spec = _spec(case["stack"], 4 if case["fp8"] else 0)
    decode = case["what"] == "decode"
    pages = sum(-(-(n + 1) // BLOCK) for n in lengths)
    cfg = _Config(
        model=spec.name, max_num_seqs=max(len(lengths), 4),
        max_model_len=MAX_LEN, num_gpu_blocks=pages + 2 + pages // 64,
        quant="fp8" if case["fp8"] else None,
        kv_dtype="fp8" if case["fp8"] else "bfloat16",
        graph_batch_sizes=tuple(
            b for b in EngineConfig.graph_batch_sizes
            if b >= len(lengths))[:1] if decode else (),
        prefill_graph_sizes=tuple(
            t for t in EngineConfig.prefill_graph_sizes
            if t >= lengths[0])[:1]
        if not decode and len(lengths) == 1 else ())
    cfg.stack = spec
    eng = LLMEngine(cfg, device="cuda:0")
    gen = torch.Generator(device="cuda:0").manual_seed(11)
    _like_trained(eng.runner.model, spec, gen, "cuda:0")
    eng.capture_graphs()
    return eng


def prepare(case, seed):
    gen = torch.Generator(device="cuda:0").manual_seed(seed)
    if case["what"] == "sample":
        return _prepare_sample(case, gen)
    lengths = _lengths(case)
    eng = _engine(case, lengths)
    decode = case["what"] == "decode"
    ids = torch.randint(0, eng.runner.spec.vocab_size,
                        (sum(lengths) + len(lengths),), generator=gen,
                        device="cuda:0").tolist()
    prompts, at = [], 0
    for n in lengths:
        prompts.append(ids[at:at + n + decode])
        at += n + decode
    state = {"engine": eng, "prompts": prompts, "lengths": lengths}
    if not decode:
        return state
    # sequences whose tokens before the last one are in the pages
    sched, runner = eng.scheduler, eng.runner
    reqs = [Request(f"s{i}", p, SamplingParams())
            for i, p in enumerate(prompts)]
    sched.schedule_portions([(r, n) for r, n in zip(reqs, lengths)])
    for pages in runner.kv_caches:
        if pages.dtype == torch.bfloat16:
            pages.normal_(generator=gen)
        else:
            for part in pages.flatten(0, 1).split(4096):
                part.copy_(torch.randn(part.shape, generator=gen,
                                       device=part.device))
    state["batch"] = ScheduledBatch("decode", reqs, len(reqs))
    state["rows"] = np.array([runner.block_manager.row_of[r.request_id]
                              for r in reqs])
    state["before"] = np.array(lengths)
    return state


def _prepare_sample(case, gen):
    b, v = case["batch"], case["vocab"]
    # next-token logits: a few dozen likely tokens far above the others
    logits = torch.randn(b, v, generator=gen, device="cuda:0")
    likely = torch.randint(0, v, (b, 48), generator=gen, device="cuda:0")
    high = 21 + 1.5 * torch.randn(b, 48, generator=gen, device="cuda:0")
    logits.scatter_(1, likely, high)
    # users set a temperature, most of them also top-p, some top-k; some
    # decode greedily
    kind = torch.arange(b, device="cuda:0") % 8
    temperature = torch.tensor([.7, 1., .8, 1., .6, .9, 0., .7],
                               device="cuda:0")[kind]
    top_p = torch.tensor([.9, 1., .95, .9, .8, 1., 1., .95],
                         device="cuda:0")[kind]
    top_k = torch.tensor([0, 0, 40, 0, 0, 50, 0, 0], dtype=torch.int32,
                         device="cuda:0")[kind]
    return {"sample": (logits.bfloat16(), temperature, top_p, top_k,
                       torch.rand(b, generator=gen, device="cuda:0"))}


# ---------------------------------------------------------------- the pass

def run(state):
    """The logits, and the pages of the last layer as the step leaves them."""
    if "sample" in state:
        return ops.sample(*state["sample"])
    eng = state["engine"]
    sched, runner = eng.scheduler, eng.runner
    if "batch" in state:
        # a decode step; its tokens are drafts that are not kept, so that the
        # next step is as long as this one
        logits = runner.forward(state["batch"])
        runner.block_manager.tokens_np[state["rows"]] = state["before"]
        return {"logits": logits, "pages": runner.kv_caches[-1]}
    # prompts in order, a step full of tokens at a time
    reqs = [Request(f"p{i}", p, SamplingParams())
            for i, p in enumerate(state["prompts"])]
    out, waiting = [], list(reqs)
    while waiting:
        portions, room = [], BUDGET
        while waiting and room:
            left = waiting[0].num_prompt_tokens - waiting[0].num_computed_tokens
            n = min(left, room)
            portions.append((waiting[0], n))
            room -= n
            if n < left:
                break
            waiting.pop(0)
        out.append(runner.forward(sched.schedule_portions(portions)))
    for r in reversed(reqs):
        sched.release(r)
    return {"logits": out, "pages": runner.kv_caches[-1]}


# ---------------------------------------------------------------- what it is

def work(case):
    if case["what"] == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": 2.0 * n, "flops": 4.0 * n}
    spec = _spec(case["stack"], 4 if case["fp8"] else 0)
    w, d = spec.hidden_size, spec.head_dim
    attn = w * (spec.num_heads + 2 * spec.num_kv_heads) * d \
        + spec.num_heads * d * w
    ff = 3 * w * spec.intermediate_size
    lengths = _lengths(case)
    decode = case["what"] == "decode"
    tokens = len(lengths) if decode else sum(lengths)
    if spec.is_moe:
        e, k = spec.num_experts, spec.num_experts_per_tok
        ff_read = ff * e * (1 - (1 - k / e) ** tokens) + e * w
        ff_used = ff * k + e * w
    else:
        ff_read = ff_used = ff
    size = 1 if case["fp8"] else 2
    kv = 2 * spec.num_kv_heads * d
    seen = sum(n + 1 for n in lengths) if decode \
        else sum(n * (n + 1) // 2 for n in lengths)
    cached = sum(lengths) if decode else 0
    layers = spec.num_layers
    return {
        "bytes": layers * (size * (attn + ff_read)
                           + size * kv * (cached + tokens))
        + 2.0 * spec.vocab_size * (w + len(lengths)) + 2.0 * tokens * w,
        "flops": layers * (2.0 * tokens * (attn + ff_used)
                           + 4.0 * spec.num_heads * d * seen)
        + 2.0 * spec.vocab_size * w * len(lengths)}


def tolerance(case):
    if case["what"] == "sample":
        # a draw falls on the boundary of two tokens
        return {"differ": 0.01}
    # bf16 activations through the layers; with 8 bits a value that lies
    # between two of their steps may take the other one
    return {"rel": 0.03, "max": 0.3} if case["fp8"] \
        else {"rel": 0.02, "max": 0.2}


# ------------------------------------------------------- in 64 bits

def _norm(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _turn(x, pos, theta):
    half = x.shape[-1] // 2
    inv = theta ** (-torch.arange(half, device=x.device).double() / half)
    ang = pos.double()[:, None, None] * inv
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(),
                      b * ang.cos() + a * ang.sin()], -1)


def _attend(q, k, v, scale):
    """q [n, H, D] are the last n positions of k, v [m, KV, D]."""
    n, m, group = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    out = torch.empty_like(q)
    at = torch.arange(m - n, m, device=q.device)
    for h in range(q.shape[1]):
        kh, vh = k[:, h // group].t().contiguous(), v[:, h // group]
        for a in range(0, n, 4096):
            s = (q[a:a + 4096, h] @ kh) * scale
            s.masked_fill_(torch.arange(m, device=q.device)[None]
                           > at[a:a + 4096, None], float("-inf"))
            out[a:a + 4096, h] = s.softmax(-1) @ vh
    return out


def _weight(layer):
    w = layer.weight.double()
    return w * layer.weight_scale.double()[:, None] \
        if layer.weight.dtype != torch.bfloat16 else w


def _experts(moe, h, spec):
    share, choice = (h @ moe.router.double().t()).softmax(-1).topk(
        spec.num_experts_per_tok, -1)
    share = share / share.sum(-1, keepdim=True)
    out = torch.zeros_like(h)
    for e in range(spec.num_experts):
        row, place = (choice == e).nonzero(as_tuple=True)
        w13, w2 = moe.w13[e].double(), moe.w2[e].double()
        if moe.w13.dtype != torch.bfloat16:
            w13 = w13 * moe.w13_scale[e].double()[:, None]
            w2 = w2 * moe.w2_scale[e].double()[:, None]
        gate, up = (h[row] @ w13.t()).chunk(2, -1)
        y = (torch.nn.functional.silu(gate) * up) @ w2.t()
        out.index_add_(0, row, y * share[row, place, None])
    return out


def _exact_sample(state):
    logits, temperature, top_p, top_k, uniform = state["sample"]
    out = []
    for b in range(logits.shape[0]):
        row = logits[b].double()
        if temperature[b] == 0:
            out.append(row.argmax())
            continue
        row = row / temperature[b].double()
        if top_k[b] > 0:
            row[row < row.topk(int(top_k[b])).values[-1]] = float("-inf")
        if top_p[b] < 1:
            p, at = row.softmax(-1).sort(descending=True)
            row[at[p.cumsum(-1) - p >= top_p[b].double()]] = float("-inf")
        c = row.softmax(-1).cumsum(-1)
        out.append((c > uniform[b].double() * c[-1]).long().argmax())
    return torch.stack(out)


def exact(case, seed):
    state = prepare(case, seed)
    if "sample" in state:
        return _exact_sample(state)
    eng = state["engine"]
    runner, spec = eng.runner, eng.runner.spec
    model, lengths = runner.model, state["lengths"]
    decode = "batch" in state
    dev = model.embed.device
    if decode:
        ids = torch.tensor([p[-1] for p in state["prompts"]], device=dev)
        pos = torch.tensor(lengths, device=dev)
        part = [1] * len(lengths)
    else:
        ids = torch.tensor(sum(state["prompts"], []), device=dev)
        pos = torch.cat([torch.arange(n, device=dev) for n in lengths])
        part = lengths
    nh, kv, d = spec.num_heads, spec.num_kv_heads, spec.head_dim
    if decode:
        tables = [torch.tensor(runner.block_manager.table(f"s{j}"),
                               device=dev) for j in range(len(part))]
        slot = torch.stack([t[n // BLOCK] * BLOCK + n % BLOCK
                            for t, n in zip(tables, lengths)])
    else:                           # pages are given out in order
        first = np.cumsum([0] + [-(-n // BLOCK) for n in lengths])
        slot = torch.cat([int(f) * BLOCK + torch.arange(n, device=dev)
                          for f, n in zip(first, lengths)])
    x = model.embed[ids].double()
    for i, layer in enumerate(model.layers):
        h = _norm(x, spec.rms_eps) * layer.input_norm_w.double()
        qkv = h @ _weight(layer.attn.qkv).t()
        q, k, v = (t.reshape(t.shape[0], -1, d) for t in
                   qkv.split([nh * d, kv * d, kv * d], -1))
        q, k = (_turn(t, pos, spec.rope_theta) for t in (q, k))
        o, at = [], 0
        for j, n in enumerate(part):
            kj, vj = k[at:at + n], v[at:at + n]
            if decode:
                old = runner.kv_caches[i][:, tables[j]].double()
                old = old.transpose(2, 3).reshape(2, -1, kv, d)
                kj = torch.cat([old[0, :lengths[j]], kj])
                vj = torch.cat([old[1, :lengths[j]], vj])
            o.append(_attend(q[at:at + n], kj, vj, d ** -0.5))
            at += n
        x = x + torch.cat(o).reshape(x.shape[0], -1) \
            @ _weight(layer.attn.o_proj).t()
        h = _norm(x, spec.rms_eps) * layer.post_norm_w.double()
        if spec.is_moe:
            x = x + _experts(layer.mlp.moe, h, spec)
        else:
            gate, up = (h @ _weight(layer.mlp.gate_up).t()).chunk(2, -1)
            x = x + (torch.nn.functional.silu(gate) * up) \
                @ _weight(layer.mlp.down).t()
    x = _norm(x, spec.rms_eps) * model.final_norm_w.double()
    head = model.lm_head.double().t()
    pages = runner.kv_caches[-1].double()
    pages[0, slot // BLOCK, :, slot % BLOCK] = k
    pages[1, slot // BLOCK, :, slot % BLOCK] = v
    if decode:
        return {"logits": x @ head, "pages": pages}
    # the last token of every portion, step by step
    out, last, done, room = [], [], 0, BUDGET
    for n in lengths:
        end = done + n
        while done < end:
            take = min(end - done, room)
            done, room = done + take, room - take
            last.append(done - 1)
            if room == 0:
                out.append(x[last] @ head)
                last, room = [], BUDGET
    if last:
        out.append(x[last] @ head)
    return {"logits": out, "pages": pages}
