"""Staged values of a decode step as a captured step reads them."""

import pytest
import torch

import hyperspot.engine  # noqa: F401  (before the models, which it imports)
import hyperspot.ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("state", [False, True])
@pytest.mark.parametrize("rows,bucket,cap,pages,width", [
    (1, 1, 4, 1, 1), (3, 4, 7, 5, 257), (4, 4, 4, 256, 256), (0, 2, 3, 0, 9)])
def test_decode_inputs(rows, bucket, cap, pages, width, state):
    g = torch.Generator().manual_seed(rows)
    stage = torch.randint(0, 1 << 20, (5 * cap + (cap * width + 1) // 2,),
                          generator=g)
    long = lambda: torch.full((bucket,), 77, device="cuda:0")
    io = {"input_ids": long(), "positions": long(), "slot_mapping": long(),
          "seq_lens": long().int(),
          "block_tables": torch.full((bucket, width), 77, device="cuda:0",
                                     dtype=torch.int32)}
    if state:
        io["state_slots"] = long().int()
    ops.decode_inputs(stage.to("cuda:0"), rows, cap, pages, io)
    names = ["input_ids", "positions", "slot_mapping", "seq_lens"] \
        + ["state_slots"] * state
    for i, (name, pad) in enumerate(zip(names, [0, 0, -1, 1, -1])):
        want = stage[i * cap:i * cap + rows].tolist() + [pad] * (bucket - rows)
        assert io[name].tolist() == want, name
    table = torch.zeros(bucket, width, dtype=torch.int32)
    table[:rows, :pages] = stage[5 * cap:].view(torch.int32)[
        :rows * pages].view(rows, pages)
    assert torch.equal(io["block_tables"].cpu(), table)
