"""Designs with states or latents at the captured steps between two prompt sizes:
logits and what a prompt leaves behind, against a pass that is not captured."""

import pytest
import torch

import mutusun_util
import radenex_util
import sumosun_util
import tefezen_util
from hyperspot import ops
from hyperspot.engine import EngineConfig, LLMEngine, SamplingParams
from hyperspot.engine.request import Request

pytestmark = pytest.mark.gpu
SIZES = (128, 264, 1000)        # of which eighths are no multiples of a tile


def setup_module():
    assert ops.have_native()


def _written(family, dtype, folder):
    if family == "mutusun":
        from test_mutusun_gpu import all_chosen
    elif family == "tefezen":
        from test_tefezen_gpu import all_chosen
    else:
        all_chosen = lambda cfg: cfg
    U = globals()[family + "_util"]
    cfg = U.standard()
    if dtype == "bfloat16":     # a last bit decides between two experts
        cfg = all_chosen(cfg)
    return U, cfg, U.write(folder, cfg, U.weights(cfg, seed=1))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("family", ["mutusun", "radenex", "sumosun", "tefezen"])
def test_prompts_of_the_steps_between(family, dtype, tmp_path):
    """The bounds are those of the sizes themselves, in the families' tests."""
    U, cfg, folder = _written(family, dtype, tmp_path)
    outs = []
    for eager in (False, True):
        eng = LLMEngine(EngineConfig(
            model=folder, dtype=dtype, max_num_seqs=4, max_model_len=1024,
            max_num_batched_tokens=1024, num_gpu_blocks=128, enforce_eager=eager,
            graph_batch_sizes=(1,), prefill_graph_sizes=SIZES), device="cuda")
        eng.capture_graphs()
        assert sorted(eng.runner._pgraphs) == (
            [] if eager else [128, 192, 224, 264, 640, 768, 1000])
        got = []
        for rep in range(3):
            for n in (129, 191, 192, 193, 224, 225, 264, 5, 639, 641, 768, 1000):
                toks = U.tokens(n + 1, cfg["vocab"], seed=n)
                req = Request(f"{rep}-{n}", toks[:n], SamplingParams())
                for tail in (n, 1):
                    batch = eng.scheduler.schedule_portions([(req, tail)])
                    got.append(eng.runner.forward(batch).float().cpu().clone())
                    req.prompt_token_ids.append(toks[n])
                eng.scheduler.release(req)
        outs.append(torch.cat(got))
        del eng
    assert U.error(outs[0], outs[1].double()) < (
        1e-5 if dtype == "float32" else 3e-2 if family == "radenex" else 2e-2)
