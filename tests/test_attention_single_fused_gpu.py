"""Attention of single tokens behind short contexts that norms, rotates and writes the cache itself, at every kind of size that the kernel takes so: float32 heads in steps of
32, more heads a KV head than a tile of sixteen holds (several workgroups norm the new key, one writes it), and with what else joins the scores.  Against the
kernel that prepares queries and keys, and 64-bit attention behind it.  Bounds as in the tests of the other start."""
import pytest
import torch

from test_attention_single_gpu import CONTEXTS, TOL, Ctx, exact, pool, staged_plan

pytestmark = pytest.mark.gpu
SIZES = [(4, 2, 32, 16), (4, 4, 96, 48), (6, 2, 160, 16), (3, 1, 224, 16), (40, 2, 128, 16), (34, 2, 64, 32), (17, 1, 64, 16), (40, 2, 96, 16), (16, 8, 128, 16)]


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_q, n_kv, d, page", SIZES)
@pytest.mark.parametrize("extra", ["plain", "softcap", "chunk and window", "sinks and gates"])
def test_fused_start(ops, dtype, n_q, n_kv, d, page, extra):
    if not ops.single_token_fusion_fits(dtype, d, page):
        assert dtype == torch.bfloat16 and d % 64
        return
    print(f"single tokens fused {dtype} {n_q}/{n_kv} d{d} page {page} {extra}", flush=True)
    torch.manual_seed(n_q + d + page)
    rows = len(CONTEXTS)
    softcap, chunk, window = 2.0 if extra == "softcap" else None, 48 if "chunk" in extra else None, 40 if "window" in extra else None
    sinks = torch.randn(n_q, device="cuda") if "sinks" in extra else None
    gates = torch.randn(rows, n_q + 3, device="cuda").to(dtype)[:, 1:1 + n_q] if "gates" in extra else None
    keys, values, table, exact_rows = pool(dtype, n_kv, d, page, CONTEXTS)
    qkv = torch.randn(rows, (n_q + 2 * n_kv) * d, device="cuda").to(dtype)
    t = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    positions, order = t([c - 1 for c in CONTEXTS]), t(list(range(rows)))
    qw, kw = 1 + 0.2 * torch.randn(d, device="cuda"), 1 + 0.2 * torch.randn(d, device="cuda")
    cos_sin = ops.rotary_table(positions, (1.0 / (1e6 ** (torch.arange(0, d, 2).float() / d))).cuda())
    ready, ready_k, ready_v = qkv.clone(), keys.clone(), values.clone()
    ops.qk_norm_rope_kv_write(ready, ready_k, ready_v, table, order, positions, qw, kw, 1e-6, cos_sin, page, n_q, n_kv, d, True)
    for r, c in enumerate(CONTEXTS):
        at, slot = int(table[r, (c - 1) // page]), (c - 1) % page
        exact_rows[r][0][c - 1], exact_rows[r][1][c - 1] = ready_k[at, :, slot].double(), ready_v[at, :, :, slot].double()
    want = exact(ready[:, :n_q * d].view(rows, n_q, d), exact_rows, d ** -0.5, window, softcap, chunk, None, sinks, gates)
    plan = staged_plan(CONTEXTS, n_q // n_kv, n_kv, window, chunk)
    for write, k, v in ((True, keys.clone(), values.clone()), (False, ready_k.clone(), ready_v.clone())):
        raw, got = qkv.clone(), torch.full((rows, n_q * d), float("nan"), device="cuda", dtype=dtype)
        ops.paged_attention(raw, got, k, v, table, order, t([1] * rows), t(CONTEXTS), plan, d ** -0.5, window, page, n_q, n_kv, d, Ctx(),
                            decode_fusion=(qw, kw, 1e-6, cos_sin, write), softcap=softcap, chunk=chunk, sinks=sinks, gates=gates)
        assert torch.equal(raw, qkv)
        torch.testing.assert_close(got.double(), want, **TOL[dtype])
        there = ~torch.isnan(ready_k)
        assert torch.equal(there, ~torch.isnan(k)) and torch.equal(torch.isnan(ready_v), torch.isnan(v)) and torch.equal(ready_v[~torch.isnan(v)], v[~torch.isnan(v)])
        torch.testing.assert_close(k[there].float(), ready_k[there].float(), **TOL[dtype])


def test_who_may_not_have_the_fused_start(ops):
    """float32 rows that are not in order: the message names what it takes."""
    contexts, n_q, n_kv, d = [5, 9], 4, 2, 64
    keys, values, table, _ = pool(torch.float32, n_kv, d, 16, contexts)
    qkv, t = torch.randn(2, (n_q + 2 * n_kv) * d, device="cuda"), lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    weight, cos_sin = torch.ones(d, device="cuda"), torch.ones(2, d, device="cuda")
    with pytest.raises(ValueError, match="rows_in_order.*float32.*got torch.float32, heads of 64, pages of 16"):
        ops.paged_attention(qkv, torch.empty(2, n_q * d, device="cuda"), keys, values, table, t([0, 1]), t([1, 1]), t(contexts), {**staged_plan(contexts, 2, n_kv), "rows_in_order": False},
                            d ** -0.5, None, 16, n_q, n_kv, d, Ctx(), decode_fusion=(weight, weight, 1e-6, cos_sin, True))
