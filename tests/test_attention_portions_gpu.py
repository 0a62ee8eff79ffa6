"""Portions of prompts, 32 pairs a wavefront: edges of its blocks, trips and pages against 64 bits, with values that are no numbers wherever the
requests have nothing."""
import numpy as np
import pytest
import torch

from llmserver_amd.parts import attention as attention_module
from llmserver_amd.parts.attention import build_attention_plan

DEV = "cuda"


class Ctx:
    def empty(self, shape, dtype=torch.bfloat16):
        return torch.empty(shape, dtype=dtype, device=DEV)


@pytest.mark.gpu
@pytest.mark.parametrize("spread", [0.3, 3.0])
@pytest.mark.parametrize("n_q,n_kv,d,page,window,walk", [(8, 2, 128, 16, None, None), (4, 4, 128, 32, 70, None), (5, 1, 64, 24, None, 6), (6, 2, 80, 16, None, 5),
                                                         (2, 2, 16, 8, 33, None), (12, 4, 96, 16, None, 3), (2, 1, 192, 16, None, 7), (4, 1, 256, 40, 100, None)])
def test_portions_against_64_bits(monkeypatch, n_q, n_kv, d, page, window, walk, spread):
    """Rows of one token behind, at and in front of the ends of blocks of 32 keys, trips of 64 and tables of 64 pages; wavefronts with one pair, none, and
    all of theirs; flat scores, and scores whose largest weights decide.  The result's own rounding is 2^-9 of a value at most and the weights' roundings
    weigh no more (independent, in a sum that is not smaller than the largest of them): 2-norms differ by less than 2^-8."""
    from llmserver_amd.kernels import default_ops
    ops, group, dtype = default_ops(), n_q // n_kv, torch.bfloat16
    _, per_tile, _ = attention_module.group_tiling(group)
    lens = [8 * per_tile + 1, 16 * per_tile, 2 * per_tile, 31, 333]
    ctxs = [8 * per_tile + 1, 64 * page + 16 * per_tile + 1, 65 * page - 1, 1024 + 31, 333 + 63]
    torch.manual_seed(n_q * d + page)
    blocks = [-(-c // page) for c in ctxs]
    keys = torch.full((sum(blocks) + 3, n_kv, page, d), float("nan"), device=DEV, dtype=dtype)
    values = torch.full((sum(blocks) + 3, n_kv, d, page), float("nan"), device=DEV, dtype=dtype)
    order = torch.randperm(sum(blocks) + 3).tolist()
    table = torch.full((len(lens), max(blocks)), -1, dtype=torch.int32)
    q = (spread * torch.randn(sum(lens), n_q * d, device=DEV)).to(dtype)
    starts, want = np.cumsum([0] + lens[:-1]), []
    for row, context in enumerate(ctxs):
        table[row, :blocks[row]] = torch.tensor([order.pop() for _ in range(blocks[row])], dtype=torch.int32)
        k, v = (torch.randn(context, n_kv, d, device=DEV).to(dtype) for _ in range(2))
        place = torch.arange(context)
        pages = table[row].long()[place // page].to(DEV)
        keys[pages, :, (place % page).to(DEV), :] = k
        values[pages, :, :, (place % page).to(DEV)] = v
        position, key = torch.arange(context - lens[row], context, device=DEV)[:, None], torch.arange(context, device=DEV)[None]
        seen = (key <= position) & (key > position - (window or context))
        for head in range(n_q):
            mine = q[starts[row]:starts[row] + lens[row], head * d:(head + 1) * d].double()
            scores = (mine @ k[:, head // group].double().T * d ** -0.5).masked_fill(~seen, float("-inf"))
            want.append((row, head, torch.softmax(scores, -1) @ v[:, head // group].double()))
    ints = lambda x: torch.tensor(np.asarray(x), dtype=torch.int32, device=DEV)
    for halves in sorted({1, ops.attention_tile_halves(dtype, d)}):
        with monkeypatch.context() as patch:
            patch.setattr(attention_module, "_workgroup_tiles_that_pay", lambda *args, **kwargs: (8, halves, walk))
            plan = build_attention_plan(lens, ctxs, group, n_kv, window, workgroup_tiles=ops.attention_workgroup_tiles(dtype, d, page), tile_halves=halves,
                                        tuning=ops.attention_tuning_for(dtype, d), tile_key_ranges=ops.attention_tile_key_ranges(dtype, d))
        assert len(plan.tiles) and plan.tiles_per_workgroup == 8 and (plan.tile_slots is not None) == (walk is not None)
        staged = {name: torch.from_numpy(getattr(plan, name)).to(DEV) for name in ("items", "item_slot", "merges", "tiles")}
        staged.update(n_tiles=len(plan.tiles), n_items=len(plan.items), n_merges=len(plan.merges), n_slots=plan.n_slots, tiles_per_workgroup=8,
                      tile_halves=halves, merge_in_workgroup=0)
        if plan.tile_slots is not None:
            staged["tile_slots"] = torch.from_numpy(plan.tile_slots).to(DEV)
        out = torch.full((sum(lens), n_q * d), float("nan"), device=DEV, dtype=dtype)
        print(f"portions {n_q} on {n_kv} of {d}, pages of {page}, window {window}, walk {walk}, {halves} halves", flush=True)
        ops.paged_attention(q, out, keys, values, table.to(DEV), ints(starts), ints(lens), ints(ctxs), staged, d ** -0.5, window, page, n_q, n_kv, d, Ctx())
        torch.cuda.synchronize()
        for row, head, exact in want:
            got = out[starts[row]:starts[row] + lens[row], head * d:(head + 1) * d].double()
            assert (got - exact).norm() < 2 ** -8 * exact.norm(), (row, head, float((got - exact).norm() / exact.norm()))


def test_captured_portions_in_large_workgroups():
    """Work lists of eight tiles a workgroup: one shape, every range of every tile in a slot of its own."""
    lens, ctx, per_tile = [37, 0, 155], [2000, 0, 155], 4
    groups, ranges = attention_module.fixed_workgroup_shape(192, 3, 4, 2, 8192, attention_module.DEFAULT_TUNING, 8)
    assert (groups, ranges) == (9, 14)
    plan = attention_module.fixed_workgroup_plan(lens, ctx, 4, None, None, groups, ranges, 192 // per_tile + 3, attention_module.DEFAULT_TUNING, 8, 2)
    assert plan.tiles_per_workgroup == 8 and plan.tile_halves == 2 and len(plan.tiles) == groups * ranges and plan.n_slots == groups * 8 * ranges
    written = {first + tile * stride for (_, q0, _, _), (first, stride) in zip(plan.tiles.tolist(), plan.tile_slots.tolist()) for tile in range(8)}
    assert {first + s for _, _, first, count in plan.merges.tolist() for s in range(count)} <= written
