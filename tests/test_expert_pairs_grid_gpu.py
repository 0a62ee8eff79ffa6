"""Experts pair by pair in launches of more than 2^24 workgroups (4,096 tokens, 8 experts each, blocks of 16 of 8,200 columns): they are taken, and every token gets what it
gets in a launch of its own few, number for number."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_more_workgroups_than_one_dimension_holds():
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    tokens, top, experts, inter, width = 4096, 8, 9, 8200, 8
    assert tokens * top * (-(-inter // 16)) > 1 << 24
    print(f"expert pairs {tokens} {top} {inter}", flush=True)
    g = torch.Generator("cuda").manual_seed(5)
    x, gate_up = (torch.randn(*shape, device="cuda", generator=g).bfloat16() for shape in ((tokens, width), (experts, 2 * inter, width)))
    chosen = torch.rand(tokens, experts, device="cuda", generator=g).topk(top, dim=1).indices.int().contiguous()
    hidden = torch.full((tokens * top, inter), float("nan"), device="cuda", dtype=torch.bfloat16)
    ops.experts_gate_up(x, gate_up, chosen, hidden)
    assert not torch.isnan(hidden).any()
    for first in (0, 2043, tokens - 5):
        few = torch.empty(5 * top, inter, device="cuda", dtype=torch.bfloat16)
        ops.experts_gate_up(x[first:first + 5], gate_up, chosen[first:first + 5].contiguous(), few)
        assert torch.equal(few, hidden[first * top:(first + 5) * top])
