"""A product that stays in parts of K for the norm is not seen outside the
model: hooks, replaced modules and direct calls have tensors."""

import pytest
import torch

from hyperspot.engine import EngineConfig, LLMEngine
import hyperspot.ops as ops
from hyperspot.models.llama import ForwardMeta


@pytest.fixture
def model(monkeypatch):
    """On the CPU, with every product that may be left in parts left in two."""
    add = ops.fused_add_rmsnorm
    monkeypatch.setattr(ops, "linear_parts", lambda x, w: ops.Parts(
        torch.stack([(x @ w.t()).float(), torch.zeros(len(x), len(w))])))
    monkeypatch.setattr(ops, "fused_add_rmsnorm", lambda x, r, *a: add(
        x.data.sum(0).to(r.dtype) if isinstance(x, ops.Parts) else x, r, *a))
    return LLMEngine(EngineConfig(
        model="tiny-llama", max_num_seqs=2, max_num_batched_tokens=64,
        max_model_len=64, num_gpu_blocks=16)).runner


def _inputs(runner, n=5):
    meta = ForwardMeta("prefill", torch.arange(n), torch.arange(n),
                       seq_start=torch.tensor([0, n], dtype=torch.int32))
    return torch.arange(n) + 3, meta, runner.kv_caches


def test_parts_are_what_the_model_adds_up(model, monkeypatch):
    ref = model.model(*_inputs(model))
    seen = []
    add = ops.fused_add_rmsnorm
    monkeypatch.setattr(ops, "fused_add_rmsnorm", lambda x, *a: (
        seen.append(type(x)), add(x, *a))[1])
    assert torch.equal(model.model(*_inputs(model)), ref)
    assert set(seen) == {ops.Parts}


@pytest.mark.parametrize("path", ["", "attn", "mlp", "attn.o_proj",
                                  "mlp.down"])
@pytest.mark.parametrize("kind", ["after", "before", "replaced", "forward",
                                  "global"])
def test_watched_modules_are_called(model, path, kind):
    layer = model.model.layers[0]
    ref = model.model(*_inputs(model))
    target, seen = layer.get_submodule(path), []

    def look(module, args, out=None):
        if module is target and out is not None:
            seen.append(out[0] if path == "" else out)
        elif module is target:
            seen.append(args[0])

    undo = None
    if kind == "after":
        target.register_forward_hook(look)
    elif kind == "before":
        target.register_forward_pre_hook(look)
    elif kind == "global":
        undo = torch.nn.modules.module.register_module_forward_hook(look)
    elif kind == "forward":
        inner = target.forward
        target.forward = lambda *a: (seen.append(a[0]), inner(*a))[1]
    else:
        class Around(torch.nn.Module):
            def __init__(self, inner):
                super().__init__()
                self.inner = inner

            def __getattr__(self, name):
                try:
                    return super().__getattr__(name)
                except AttributeError:
                    return getattr(self.inner, name)

            def forward(self, *args):
                out = self.inner(*args)
                seen.append(out[0] if path == "" else out)
                return out

        if path == "":
            model.model.layers[0] = Around(target)
        else:
            owner, _, name = path.rpartition(".")
            setattr(layer.get_submodule(owner), name, Around(target))
    try:
        out = model.model(*_inputs(model))
    finally:
        if undo:
            undo.remove()
    assert len(seen) == 1 and isinstance(seen[0], torch.Tensor)
    assert torch.equal(out, ref)


def test_direct_calls_give_tensors(model):
    layer, (ids, meta, caches) = model.model.layers[0], _inputs(model)
    x = model.model.embed[ids]
    cs = model.model.cos_sin
    assert isinstance(layer.attn(x, meta, caches[0], cs), torch.Tensor)
    assert isinstance(layer.mlp(x), torch.Tensor)
    h, residual = layer(x, None, meta, kv_cache=caches[0], cos_sin=cs)
    assert isinstance(h, torch.Tensor) and isinstance(residual, torch.Tensor)
