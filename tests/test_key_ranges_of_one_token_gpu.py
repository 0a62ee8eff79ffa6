"""One token behind a long context: every key range leaves a partial result of its own, one merge puts them all together; against 64 bits, over replays."""
import numpy as np
import pytest
import torch

from llmserver_amd.parts.attention import group_tiling, stage_attention_plan


@pytest.mark.gpu
@pytest.mark.parametrize("n_q,n_kv,d,window,dtype,fused", [(16, 8, 128, None, torch.bfloat16, False), (16, 8, 128, None, torch.bfloat16, True),
                                                           (16, 8, 128, None, torch.float32, False), (4, 4, 64, None, torch.bfloat16, True),
                                                           (8, 1, 64, 700, torch.bfloat16, True), (8, 1, 64, 700, torch.float32, False),
                                                           (2, 2, 256, None, torch.bfloat16, True), (20, 1, 32, None, torch.bfloat16, False)])
def test_one_token_behind_long_contexts(n_q, n_kv, d, window, dtype, fused):
    """Contexts that leave ranges empty, end at their edges and fill them.  The result is the ranges' results weighed with their maxima and sums: a rounding of 32-bit sums (2^-20
    of its norm, a hundredth of what is left to bfloat16 anyway) and, in bfloat16, its own (2^-8 of a number).  Against 64 bits: 2^-20 of the result's norm in float32; in bfloat16 the
    weights' and the result's roundings, below 2^-8.  Replays in a row give the same numbers bit by bit."""
    from llmserver_amd.engine.batch import Staging, StepContext
    from llmserver_amd.kernels import default_ops
    ops, page, most, group = default_ops(), 16, 4096, n_q // n_kv
    torch.manual_seed(n_q + d)
    keys, values = torch.randn(most // page, n_kv, page, d, device="cuda").to(dtype), torch.randn(most // page, n_kv, d, page, device="cuda").to(dtype)
    table = np.random.RandomState(d).permutation(most // page).astype(np.int32)[None]
    staging, graph = Staging("cuda", 1 << 16), None
    qkv, out = torch.zeros(1, (n_q + 2 * n_kv) * d, device="cuda", dtype=dtype), torch.zeros(1, n_q * d, device="cuda", dtype=dtype)
    weights, cos_sin = torch.ones(d, device="cuda"), torch.zeros(1, d, device="cuda")
    cos_sin[:, :d // 2] = 1.0                              # (a rotation by nothing: the fused start norms alone)
    heads_of_tile, _, group_tiles = group_tiling(group)
    for context in (most, 1, 33, 700, 2049, 4095):
        print(f"one token {dtype} fused {fused} {n_q}/{n_kv} of {d} window {window} context {context}", flush=True)
        ctx = StepContext(ops, "cuda", dtype, staging)
        ctx.page_size = page
        ctx.fill(np.zeros(1), [context - 1], np.zeros(1), np.zeros(1), np.ones(1), [context], [], [table], None, [0])
        ctx.static_max_keys = most
        stage_attention_plan(ctx, "plan", group, n_kv, d, window, lambda rows, longest: None)
        plan = ctx.get_plan("plan")
        assert plan["n_items"] == plan["n_slots"] > 4 and plan["n_merges"] == 1
        ctx.stage()
        staging.upload()
        qkv.copy_(torch.randn_like(qkv))
        flat_k = keys[torch.from_numpy(table[0]).cuda().long()].permute(1, 0, 2, 3).reshape(n_kv, most, d).double()
        flat_v = values[torch.from_numpy(table[0]).cuda().long()].permute(1, 0, 3, 2).reshape(n_kv, most, d).double()
        heads = qkv.view(n_q + 2 * n_kv, d).double()
        q = heads[:n_q]
        if fused:
            normed = lambda x: (x * (x.pow(2).mean(-1, keepdim=True) + 1e-6).rsqrt()).to(dtype).double()
            q, flat_k[:, context - 1], flat_v[:, context - 1] = normed(q), normed(heads[n_q:n_q + n_kv]), heads[n_q + n_kv:]
        first = max(0, context - window) if window else 0
        scores = torch.stack([flat_k[h // group, first:context] @ q[h] for h in range(n_q)]) * d ** -0.5
        exact = torch.stack([torch.softmax(scores[h], -1) @ flat_v[h // group, first:context] for h in range(n_q)]).reshape(1, -1)
        scratch = {}

        class Ctx:
            def empty(self, shape, dtype=dtype):
                scratch[shape[-1]] = torch.full(shape, float("nan"), device="cuda", dtype=dtype)
                return scratch[shape[-1]]

        def attend(of):
            extra = {"decode_fusion": (weights, weights, 1e-6, cos_sin, True)} if fused else {}
            ops.paged_attention(qkv, out, keys, values, ctx.block_table(0), ctx.row_start, ctx.row_len, ctx.row_ctx, plan, d ** -0.5, window, page, n_q, n_kv, d, of, **extra)
        attend(Ctx())
        torch.cuda.synchronize()
        eager = out.clone()
        # slots x (KV heads x tiles of a group) x pairs, of which a tile's first ones are its heads of the one token
        acc, ml = (scratch[last].double().view(-1, n_kv, group_tiles, 16, last)[:, :, :, :heads_of_tile].reshape(-1, n_kv, group_tiles * heads_of_tile, last)[:, :, :group]
                   .reshape(-1, n_q, last) for last in (d, 2))
        assert bool(acc.isfinite().all()) and not bool(ml.isnan().any())          # (of every range, also of those without keys)
        weight = (ml[..., 0] - ml[..., 0].amax(0)).exp()
        merged = ((weight[..., None] * acc).sum(0) / (weight * ml[..., 1]).sum(0)[:, None]).reshape(1, -1)
        off = (eager.double() - merged).abs()
        assert bool((off <= 2 ** -20 * merged.norm() + (2 ** -8 * merged.abs() if dtype == torch.bfloat16 else 0)).all())
        assert (eager.double() - exact).norm() <= (2 ** -20 if dtype == torch.float32 else 2 ** -8) * exact.norm()
        if graph is None:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                attend(ctx)
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager)
