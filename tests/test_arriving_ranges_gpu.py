"""One token's key ranges, merged by the workgroup that ends last: against 64 bits, over replays, and which steps go so."""
import numpy as np
import pytest
import torch

from llmserver_amd.parts.attention import arriving_workgroups, stage_attention_plan


def test_which_steps_go_so():
    assert arriving_workgroups(1, 128, 256) == 32 and arriving_workgroups(1, 8, 512) == 2
    assert arriving_workgroups(1, 4, 256) is None and arriving_workgroups(1, 42, 256) is None and arriving_workgroups(1, 64, 513) is None
    assert arriving_workgroups(2, 64, 256) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,fused", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float32, False)])
@pytest.mark.parametrize("n_q,n_kv,d,window", [(16, 8, 128, None), (4, 4, 64, None), (8, 1, 64, 700), (2, 2, 256, None), (32, 8, 16, None)])
def test_one_token_behind_long_contexts(dtype, fused, n_q, n_kv, d, window):
    """Contexts that leave ranges empty, end at their edges and fill them; the counters are back at zero behind every launch, and replays in a row give the
    same numbers bit by bit.  Sums of 32-bit numbers: 2^-20 of the result's norm in float32; in bfloat16 the weights' and the result's roundings, below 2^-8."""
    if fused and d % 64:
        return
    from llmserver_amd.engine.batch import Staging, StepContext
    from llmserver_amd.kernels import default_ops
    ops, page, most = default_ops(), 16, 4096
    torch.manual_seed(n_q + d)
    keys, values = torch.randn(most // page, n_kv, page, d, device="cuda").to(dtype), torch.randn(most // page, n_kv, d, page, device="cuda").to(dtype)
    table = np.random.RandomState(d).permutation(most // page).astype(np.int32)[None]
    staging, graph = Staging("cuda", 1 << 16), None
    qkv, out = torch.zeros(1, (n_q + 2 * n_kv) * d, device="cuda", dtype=dtype), torch.zeros(1, n_q * d, device="cuda", dtype=dtype)
    weights, cos_sin = torch.ones(d, device="cuda"), torch.zeros(1, d, device="cuda")
    cos_sin[:, :d // 2] = 1.0                              # (a rotation by nothing: the fused start norms alone)
    for context in (most, 1, 33, 700, 2049, 4095):
        print(f"arriving {dtype} fused {fused} {n_q}/{n_kv} of {d} window {window} context {context}", flush=True)
        ctx = StepContext(ops, "cuda", dtype, staging)
        ctx.page_size = page
        ctx.fill(np.zeros(1), [context - 1], np.zeros(1), np.zeros(1), np.ones(1), [context], [], [table], None, [0])
        ctx.static_max_keys = most
        stage_attention_plan(ctx, "plan", n_q // n_kv, n_kv, d, window, lambda rows, longest: None)
        plan = ctx.get_plan("plan")
        assert plan["workgroups_a_tile"] == plan["n_items"] // 4 >= 2
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
        scores = torch.stack([flat_k[h // (n_q // n_kv), first:context] @ q[h] for h in range(n_q)]) * d ** -0.5
        exact = torch.stack([torch.softmax(scores[h], -1) @ flat_v[h // (n_q // n_kv), first:context] for h in range(n_q)]).reshape(1, -1)

        def attend():
            extra = {"decode_fusion": (weights, weights, 1e-6, cos_sin, True)} if fused else {}
            ops.paged_attention(qkv, out, keys, values, ctx.block_table(0), ctx.row_start, ctx.row_len, ctx.row_ctx, plan, d ** -0.5, window, page, n_q, n_kv, d, ctx, **extra)
        if graph is None:
            attend()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                attend()
        seen = []
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            seen.append(out.clone())
            assert not plan["arrivals"].any()
        assert torch.equal(seen[0], seen[1]) and torch.equal(seen[0], seen[2])
        assert (seen[0].double() - exact).norm() <= (2 ** -20 if dtype == torch.float32 else 2 ** -8) * exact.norm()
