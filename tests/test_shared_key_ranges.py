"""Key ranges that a step's rows share by their lengths: arrays of one shape whatever the contexts are, every key once, no range longer than the
even cut's longest."""
import random

import numpy as np
import pytest

from llmserver_amd.parts.attention import MAX_SPLITS, build_attention_plan, first_keys


@pytest.mark.parametrize("rows, splits", [(2, 2), (2, 64), (3, 5), (33, 3), (40, 3), (7, 17), (128, 2)])
@pytest.mark.parametrize("window, chunk", [(None, None), (300, None), (None, 256)])
def test_every_key_is_read_once_and_shapes_stay(rows, splits, window, chunk):
    order = random.Random(rows * splits)
    for contexts in ([1] * rows, [4000] * rows, [order.randint(1, 4500) for _ in range(rows)], [1] * (rows - 1) + [8191], [order.choice((1, 31, 32, 33, 65)) for _ in range(rows)]):
        plan = build_attention_plan([1] * rows, contexts, 4, 8, window, fixed_splits=splits, chunk=chunk, share_ranges=True)
        even = build_attention_plan([1] * rows, contexts, 4, 8, window, fixed_splits=splits, chunk=chunk)
        assert plan.items.shape == (rows * splits, 4) == even.items.shape and plan.merges.shape == even.merges.shape == (rows, 4)
        assert plan.n_slots == rows * splits and (plan.item_slot == np.arange(rows * splits)).all() and plan.merge_in_workgroup == 0
        assert (plan.merges[:, 3] <= MAX_SPLITS).all() and (plan.merges[:, 3] >= 1).all()
        longest = lambda p: int((p.items[:, 3] - p.items[:, 2]).max())
        assert longest(plan) <= longest(even) + 31          # (a row's first range begins at a multiple of 32 keys, which a window may lie behind)
        begins = first_keys(np.asarray(contexts) - 1, window, chunk)
        for row, (of_row, q0, first, count) in enumerate(plan.merges):
            mine = plan.items[first:first + count]
            assert of_row == row and q0 == 0 and (mine[:, 0] == row).all() and (mine[:, 1] == 0).all()
            place = int(begins[row])
            for _, _, lo, hi in mine:
                assert lo <= hi and (lo == place or lo == hi == contexts[row]) and (lo % 32 == 0 or lo == begins[row] or lo == contexts[row])
                place = max(place, int(hi))
            assert place == contexts[row] and (mine[:, 3] > mine[:, 2]).any()


def test_uneven_rows_get_shorter_ranges():
    contexts = [667 + 42 * i for i in range(33)] + [1] * 7
    shared, even = (build_attention_plan([1] * 40, contexts, 4, 8, None, fixed_splits=3, share_ranges=share) for share in (True, False))
    longest = lambda p: int((p.items[:, 3] - p.items[:, 2]).max())
    assert longest(shared) == 480 and longest(even) == 672


@pytest.mark.parametrize("fused", [False, True])
def test_where_the_even_cut_is_the_better_one(fused):
    """Rows of one length and ranges that sharing does not shorten: the very plan of the even cut; where attention prepares its queries itself, also ranges
    that sharing hardly shortens or that are short already."""
    order = random.Random(7)
    plans = lambda rows, splits, contexts: [build_attention_plan([1] * rows, contexts, 4, 8, None, fixed_splits=splits, share_ranges=share, fused=fused) for share in (True, False)]
    longest = lambda p: int((p.items[:, 3] - p.items[:, 2]).max())
    for rows, splits, contexts in ((40, 3, [2000] * 40), (8, 16, [4001] * 8), (2, 32, [1300, 1400]), (4, 32, [2000, 2000, 500, 500]), (16, 8, order.sample(range(1900, 2000), 16))):
        shared, even = plans(rows, splits, contexts)
        assert np.array_equal(shared.items, even.items) and np.array_equal(shared.merges, even.merges) and shared.n_slots == even.n_slots
    for rows, splits, contexts in ((8, 16, [600, 300, 300, 300, 200, 200, 200, 200]), (16, 8, [int(900 * (15 + 2 * i) / 45) for i in range(16)])):
        shared, even = plans(rows, splits, contexts)
        assert np.array_equal(shared.items, even.items) == fused and (fused or longest(shared) <= 0.75 * longest(even))
    for rows, splits, contexts in ((24, 5, [2000] + [100] * 23), (16, 8, [int(4400 * (15 + 2 * i) / 45) for i in range(16)]), (8, 16, [1300] * 4 + [325] * 4)):
        shared, even = plans(rows, splits, contexts)
        assert longest(shared) <= 0.72 * longest(even)


def test_who_prepares_its_queries_itself():
    """Mixers say so to the plan: a plain one in the type and head sizes of the fused start, no other."""
    import types

    import torch

    from llmserver_amd.parts import attention
    from llmserver_amd.parts.rope import RotaryPosition
    asked = []
    ops = types.SimpleNamespace(decode_fusion_fits=lambda dtype, head_dim: dtype == torch.bfloat16 and head_dim % 64 == 0)
    stage, attention.stage_attention_plan = attention.stage_attention_plan, lambda *args: asked.append(args[8])
    try:
        for head_dim, dtype, general in ((64, torch.bfloat16, {}), (64, torch.float32, {}), (48, torch.bfloat16, {}), (64, torch.bfloat16, {"head_gate": True})):
            attention.GQAttention(64, 4, 2, head_dim, RotaryPosition(head_dim, 1e4), qk_norm_eps=1e-6, **general).prepare(types.SimpleNamespace(ops=ops, dtype=dtype))
    finally:
        attention.stage_attention_plan = stage
    assert asked == [True, False, False, False]
