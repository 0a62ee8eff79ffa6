"""Steps of so many rows of one token that the kernel for single tokens would not pay: they are the other kernel's again, number for number."""
import pytest
import torch

from test_attention_single_gpu import Ctx, pool, staged_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows, n_q, n_kv, d", [(70, 16, 8, 128), (66, 32, 8, 64), (33, 32, 16, 32)])
@pytest.mark.parametrize("fused", [False, True])
def test_rows_beyond_the_compute_units(dtype, rows, n_q, n_kv, d, fused):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    fused = fused and ops.decode_fusion_fits(dtype, d)
    print(f"many single tokens {dtype} {rows} rows {n_q}/{n_kv} d{d} fused {fused}", flush=True)
    torch.manual_seed(rows)
    contexts = [1 + (37 * r) % 300 for r in range(rows)]
    keys, values, table, _ = pool(dtype, n_kv, d, 16, contexts)
    qkv = torch.randn(rows, (n_q + 2 * n_kv) * d, device="cuda").to(dtype)
    t = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    weight, cos_sin = torch.ones(d, device="cuda"), torch.randn(rows, d, device="cuda")
    plan, got = staged_plan(contexts, n_q // n_kv, n_kv), []
    assert not ops.single_tokens_pay(dtype, d, rows, n_q, n_kv)
    for in_order in (True, False):
        out, k, v = torch.full((rows, n_q * d), float("nan"), device="cuda", dtype=dtype), keys.clone(), values.clone()
        extra = {"decode_fusion": (weight, weight, 1e-6, cos_sin, True)} if fused else {}
        ops.paged_attention(qkv, out, k, v, table, t(list(range(rows))), t([1] * rows), t(contexts), {**plan, "rows_in_order": in_order}, d ** -0.5, None, 16,
                            n_q, n_kv, d, Ctx(), **extra)
        got.append((out, k, v))
    assert not torch.isnan(got[0][0]).any()
    for a, b in zip(*got):
        assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
