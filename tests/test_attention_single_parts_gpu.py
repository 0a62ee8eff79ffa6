"""Attention of single tokens in few rows: workgroups that share a row's keys of a KV head, each with a part of the value's dimensions, form the same sums as
one that has all of them: equal bits with the same rows in a step of many, contexts at the edges of pages, key steps and wavefronts' rounds."""
import pytest
import torch

from test_attention_single_gpu import CONTEXTS, Ctx, pool, staged_plan

pytestmark = pytest.mark.gpu
SHAPES = [(8, 8, 128, 16), (16, 8, 128, 32), (32, 8, 128, 16), (8, 8, 64, 16), (6, 2, 64, 48), (12, 1, 128, 64), (16, 1, 256, 16), (10, 1, 192, 16), (8, 2, 96, 16)]


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_q, n_kv, d, page", SHAPES)
@pytest.mark.parametrize("extra", ["plain", "fused", "fused and written", "window", "softcap", "sinks and gates"])
def test_few_rows_and_many_give_the_same_bits(ops, dtype, n_q, n_kv, d, page, extra):
    fused = "fused" in extra
    if fused and not ops._attention_library(dtype, d).lsa_attention_single_fits(page, 1):
        pytest.skip("norm and rotation are a launch of their own at this head size")
    print(f"single tokens shared {dtype} {n_q}/{n_kv} d{d} page {page} {extra}", flush=True)
    torch.manual_seed(n_q * d + page)
    contexts = (CONTEXTS * 4)[:max(len(CONTEXTS), 80 // n_kv)]       # (more than 64 workgroups: each has its row to itself)
    keys, values, table, _ = pool(dtype, n_kv, d, page, contexts)
    qkv = torch.randn(len(contexts), (n_q + 2 * n_kv) * d, device="cuda").to(dtype)
    window, softcap = 40 if extra == "window" else None, 2.0 if extra == "softcap" else None
    sinks = torch.randn(n_q, device="cuda") if "sinks" in extra else None
    gates = torch.randn(len(contexts), n_q, device="cuda").to(dtype) if "gates" in extra else None
    t = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    qw, kw = 1 + 0.2 * torch.randn(d, device="cuda"), 1 + 0.2 * torch.randn(d, device="cuda")
    cos_sin = ops.rotary_table(t([c - 1 for c in contexts]), (1.0 / (1e6 ** (torch.arange(0, d, 2).float() / d))).cuda())

    def attend(first, last, k, v):
        some, rows = contexts[first:last], last - first
        got = torch.full((rows, n_q * d), float("nan"), device="cuda", dtype=dtype)
        fusion = (qw, kw, 1e-6, cos_sin[first:last].contiguous(), extra == "fused and written") if fused else None
        ops.paged_attention(qkv[first:last].contiguous(), got, k, v, table[first:last].contiguous(), t(list(range(rows))), t([1] * rows), t(some),
                            staged_plan(some, n_q // n_kv, n_kv, window), d ** -0.5, window, page, n_q, n_kv, d, Ctx(), decode_fusion=fusion, sinks=sinks, softcap=softcap,
                            gates=gates[first:last] if gates is not None else None)
        return got

    many_k, many_v, few_k, few_v = keys.clone(), values.clone(), keys.clone(), values.clone()
    many = attend(0, len(contexts), many_k, many_v)
    assert not torch.isnan(many).any()
    for first in range(0, len(CONTEXTS), 4):
        assert torch.equal(attend(first, first + 4, few_k, few_v), many[first:first + 4])
    for first in range(len(CONTEXTS), len(contexts), 4):
        attend(first, first + 4, few_k, few_v)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    assert torch.equal(few_k.view(bits), many_k.view(bits)) and torch.equal(few_v.view(bits), many_v.view(bits))
