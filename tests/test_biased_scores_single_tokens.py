"""Attention with query and key norms, a rotation and a bias by distance, in steps of one token a row behind short contexts: the kernels that do norm and rotation inside attention
know no bias, so these come in front of it, whatever kernels fit the type and the head size."""
import types

import pytest
import torch

from llmserver_amd.parts.attention import GQAttention
from llmserver_amd.parts.rope import RotaryPosition


@pytest.mark.parametrize("merge", [0, 4])
@pytest.mark.parametrize("biased", [True, False])
def test_norm_and_rotation_come_in_front_of_biased_scores(merge, biased):
    calls = []
    ops = types.SimpleNamespace(
        decode_fusion_fits=lambda dtype, head_dim: True, single_token_fusion_fits=lambda *sizes: True,
        qk_norm_rope_kv_write=lambda *args: calls.append("in front"),
        paged_attention=lambda *args, **extra: calls.append(("attention", "decode_fusion" in extra, extra.get("slopes"))))
    mixer = GQAttention(64, 4, 2, 32, RotaryPosition(32, 1e4), qk_norm_eps=1e-6, distance_bias=biased)
    mixer.q_norm_weight = mixer.k_norm_weight = torch.ones(32)
    mixer.slopes = torch.ones(4) if biased else None
    mixer.qkv.forward = lambda x, ctx: torch.zeros(3, 8 * 32)
    mixer.o.forward = lambda out, ctx, sink=None: out
    mixer.position.cos_sin = lambda ctx: torch.ones(3, 32)
    ctx = types.SimpleNamespace(ops=ops, n_tokens=3, n_rows=3, row_start=None, row_len=None, row_ctx=None, token_row=None, positions=None, block_table=lambda group: None,
                                get_plan=lambda key: {"rows_in_order": True, "merge_in_workgroup": merge}, empty=lambda shape: torch.empty(shape))
    cache = types.SimpleNamespace(group=0, keys=None, values=None, page_size=16, writable=True)
    mixer.forward(torch.zeros(3, 64), ctx, cache)
    if biased:
        assert calls == ["in front", ("attention", False, mixer.slopes)]
    else:
        assert calls == [("attention", True, None)]
