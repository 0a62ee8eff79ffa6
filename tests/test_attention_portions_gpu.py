"""Portions of prompts in workgroups of as many tiles as the kernel takes: edges of steps, tiles and pages against 64 bits, with values that are no numbers wherever the
requests have nothing; and what is rounded on the way."""
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
    """Rows of one token behind, at and in front of the ends of steps of 32 keys, of pages and of tables of 64 pages; wavefronts with one pair, none, and
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
    per_workgroup = ops.attention_workgroup_tiles(dtype, d, page)
    for halves in sorted({1, ops.attention_tile_halves(dtype, d)}):
        with monkeypatch.context() as patch:
            patch.setattr(attention_module, "_workgroup_tiles_that_pay", lambda *args, **kwargs: (per_workgroup, halves, walk))
            plan = build_attention_plan(lens, ctxs, group, n_kv, window, workgroup_tiles=per_workgroup, tile_halves=halves,
                                        tuning=ops.attention_tuning_for(dtype, d), tile_key_ranges=ops.attention_tile_key_ranges(dtype, d))
        assert len(plan.tiles) and plan.tiles_per_workgroup == per_workgroup and (plan.tile_slots is not None) == (walk is not None)
        staged = {name: torch.from_numpy(getattr(plan, name)).to(DEV) for name in ("items", "item_slot", "merges", "tiles")}
        staged.update(n_tiles=len(plan.tiles), n_items=len(plan.items), n_merges=len(plan.merges), n_slots=plan.n_slots, tiles_per_workgroup=per_workgroup,
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


@pytest.mark.gpu
@pytest.mark.parametrize("per_workgroup", [4, 8])
def test_weights_are_rounded_once_and_summed_as_they_were(monkeypatch, per_workgroup):
    """Weights go into the products with the values as exp(score - the row's highest score so far) rounded to bfloat16, steps of 32 keys one behind another; what they are divided by is
    their sum before that rounding, in 32 bits.  That computed in 64 bits and rounded is what comes out, but for results as good as halfway between two numbers and for weights that
    are (an exponential is off by some 2^-23: one weight in 30,000, of 64): fewer than one result in fifty.  (Sums of rounded weights and a maximum that lags change one in twenty.)"""
    from llmserver_amd.kernels import default_ops
    ops, dtype, heads, group, d, page, n = default_ops(), torch.bfloat16, 8, 4, 128, 16, 64
    if per_workgroup > ops.attention_workgroup_tiles(dtype, d, page):
        pytest.skip("no such form")
    torch.manual_seed(7)
    q, k, v = (torch.randn(n, count, d, device=DEV).to(dtype) for count in (heads, heads // group, heads // group))
    keys = k.view(n // page, page, heads // group, d).permute(0, 2, 1, 3).contiguous()
    values = v.view(n // page, page, heads // group, d).permute(0, 2, 3, 1).contiguous()
    table = torch.arange(n // page, dtype=torch.int32, device=DEV)[None]
    with monkeypatch.context() as patch:
        patch.setattr(attention_module, "_workgroup_tiles_that_pay", lambda *args, **kwargs: (per_workgroup, 1, None))
        plan = build_attention_plan([n], [n], group, heads // group, None, workgroup_tiles=ops.attention_workgroup_tiles(dtype, d, page), tuning=ops.attention_tuning_for(dtype, d))
    assert len(plan.tiles) and plan.tiles_per_workgroup == per_workgroup
    staged = {name: torch.from_numpy(getattr(plan, name)).to(DEV) for name in ("items", "item_slot", "merges", "tiles")}
    staged.update(n_tiles=len(plan.tiles), n_items=len(plan.items), n_merges=len(plan.merges), n_slots=plan.n_slots, tiles_per_workgroup=per_workgroup, tile_halves=1,
                  merge_in_workgroup=0)
    out = torch.empty(n, heads * d, device=DEV, dtype=dtype)
    ints = lambda x: torch.tensor([x], dtype=torch.int32, device=DEV)
    print(f"weights, {per_workgroup} tiles a workgroup", flush=True)
    ops.paged_attention(q.view(n, heads * d), out, keys, values, table, ints(0), ints(n), ints(n), staged, d ** -0.5, None, page, heads, heads // group, d, Ctx())
    torch.cuda.synchronize()
    k, v = (x.double().cpu().repeat_interleave(group, dim=1) for x in (k, v))
    scores = torch.einsum("qhd,khd->hqk", q.double().cpu(), k) * d ** -0.5
    scores = scores.masked_fill(~torch.ones(n, n, dtype=torch.bool).tril(), float("-inf"))
    top, total, sums = torch.full((heads, n, 1), float("-inf"), dtype=torch.float64), 0.0, 0.0
    for at in range(0, n, 32):
        after = torch.maximum(top, scores[..., at:at + 32].amax(-1, keepdim=True))
        weights, kept = (scores[..., at:at + 32] - after).exp(), (top - after).exp()
        total = total * kept + weights.sum(-1, keepdim=True)
        sums = sums * kept + torch.einsum("hqk,khd->hqd", weights.to(dtype).double(), v[at:at + 32])
        top = after
    expected = (sums / total).permute(1, 0, 2).reshape(n, heads * d).to(dtype)
    assert float((out.cpu() != expected).double().mean()) < 0.02
