"""A captured step of single tokens whose rows get and lose key ranges between two replays (one long row among short ones, rows of one length, all lengths, the long row
elsewhere): every replay against 64 bits, with its norm, rotation and cache write in attention's fused start and without.

Bounds: float32 sums of at most 2,200 weighted values of up to 5: 5e-5; bfloat16 rounds probabilities and results to 2^-9 of values of 1 to 4: 2e-2."""
import numpy as np
import pytest
import torch

from llmserver_amd.engine.batch import Staging, StepContext
from llmserver_amd.parts.attention import stage_attention_plan
from test_attention_single_gpu import exact, pool

pytestmark = pytest.mark.gpu
TOL = {torch.float32: dict(atol=5e-5, rtol=1e-5), torch.bfloat16: dict(atol=2e-2, rtol=2e-2)}


@pytest.mark.parametrize("dtype, fused", [(torch.float32, False), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("rows, n_q, n_kv", [(24, 8, 8), (40, 16, 8), (8, 16, 8)])
def test_rows_get_and_lose_ranges_between_replays(dtype, fused, rows, n_q, n_kv):
    from llmserver_amd.kernels import default_ops
    ops, d, page, most = default_ops(), 64, 16, 2200
    print(f"shared ranges replayed {dtype} fused {fused} {rows} rows {n_q}/{n_kv}", flush=True)
    torch.manual_seed(rows)
    spread = [600 + (most - 600) * ((7 * r) % rows) // rows for r in range(rows)]
    kinds = [[most] + [90] * (rows - 1), [1500] * rows, spread, [1] * (rows - 1) + [most], spread[::-1], [513] + [1] * (rows - 1)]
    keys, values, table, stored = pool(dtype, n_kv, d, page, [most] * rows)
    kept_keys, kept_values = keys.clone(), values.clone()
    staging, graph, layouts, counts = Staging("cuda", 1 << 17), None, set(), set()
    qkv = torch.zeros(rows, (n_q + 2 * n_kv) * d, device="cuda", dtype=dtype)
    out = torch.zeros(rows, n_q * d, device="cuda", dtype=dtype)
    weights, cos_sin = torch.ones(d, device="cuda"), torch.zeros(rows, d, device="cuda")
    cos_sin[:, :d // 2] = 1.0                              # (a rotation by nothing: the fused start norms alone)
    for contexts in kinds:
        ctx = StepContext(ops, "cuda", dtype, staging)
        ctx.page_size = page
        ctx.fill(np.zeros(rows), np.asarray(contexts) - 1, np.arange(rows), np.arange(rows), np.ones(rows), contexts, [], [table.cpu().numpy()], None, list(range(rows)))
        ctx.static_max_keys = 4096
        stage_attention_plan(ctx, "plan", n_q // n_kv, n_kv, d, None, lambda r, longest: None)
        plan = ctx.get_plan("plan")
        assert plan["n_merges"] == rows and not plan["merge_in_workgroup"]
        counts.add(tuple(plan["merges"][:, 3]))
        ctx.stage()
        layouts.add(ctx.layout)
        staging.upload()
        keys.copy_(kept_keys)
        values.copy_(kept_values)
        qkv.copy_(torch.randn_like(qkv))

        def attend():
            extra = {"decode_fusion": (weights, weights, 1e-6, cos_sin, True)} if fused else {}
            ops.paged_attention(qkv, out, keys, values, ctx.block_table(0), ctx.row_start, ctx.row_len, ctx.row_ctx, plan, d ** -0.5, None, page, n_q, n_kv, d, ctx, **extra)
        if graph is None:
            attend()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                attend()
        for _ in range(2):                                 # (the program's own work between the replays: clears)
            out.zero_()
            keys.copy_(kept_keys)
            values.copy_(kept_values)
            graph.replay()
            torch.cuda.synchronize()
            q = qkv[:, :n_q * d].view(rows, n_q, d)
            seen = [(k[:c].clone(), v[:c].clone()) for (k, v), c in zip(stored, contexts)]
            if fused:
                unit = lambda x: (x.double() * torch.rsqrt(x.double().pow(2).mean(dim=-1, keepdim=True) + 1e-6)).to(dtype)
                q = unit(q)
                for r in range(rows):
                    seen[r][0][-1] = unit(qkv[r, n_q * d:(n_q + n_kv) * d].view(n_kv, d)).double()
                    seen[r][1][-1] = qkv[r, (n_q + n_kv) * d:].view(n_kv, d).double()
            torch.testing.assert_close(out.double(), exact(q, seen, d ** -0.5, None, None, None, None, None, None), **TOL[dtype])
    assert len(layouts) == 1 and len(counts) >= 3
