"""Attention of steps of one token a row behind short contexts (the kernel that finds its row by its place in the launch), against plain
64-bit attention: contexts at the edges of pages, key steps and wavefronts' rounds, tables of more than 64 pages, what else may join the
scores, and pages whose unused places hold no numbers.

Bounds: float32 results are sums of at most 1,025 weighted values, in chains of a few hundred roundings of 2^-24 of values of up to about 10:
2e-5 as in the tests beside this one; bfloat16 rounds probabilities and results to 2^-9 of values of 1 to 4: 2e-2."""
import itertools

import numpy as np
import pytest
import torch

from llmserver_amd.parts.attention import build_attention_plan

pytestmark = pytest.mark.gpu
TOL = {torch.float32: dict(atol=2e-5, rtol=1e-5), torch.bfloat16: dict(atol=2e-2, rtol=2e-2)}
CONTEXTS = [1, 2, 15, 16, 17, 31, 32, 33, 63, 127, 128, 129, 225, 255, 256, 257, 300, 511, 512, 1025]


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


class Ctx:
    def empty(self, shape, dtype=None):
        return torch.empty(shape, device="cuda", dtype=dtype)


def pool(dtype, n_kv, d, page, contexts):
    """Pages in scrambled order whose unused places are NaN, a table, and every row's keys and values in 64 bits."""
    count = sum(-(-c // page) for c in contexts) + 2
    keys = torch.full((count, n_kv, page, d), float("nan"), device="cuda", dtype=dtype)
    values = torch.full((count, n_kv, d, page), float("nan"), device="cuda", dtype=dtype)
    table = torch.full((len(contexts), max(-(-c // page) for c in contexts)), -1, dtype=torch.int32)
    order, rows = iter(torch.randperm(count).tolist()), []
    for r, c in enumerate(contexts):
        blocks = -(-c // page)
        table[r, :blocks] = torch.tensor(list(itertools.islice(order, blocks)), dtype=torch.int32)
        k, v = (torch.randn(c, n_kv, d, device="cuda").to(dtype) for _ in range(2))
        place = torch.arange(c)
        at = table[r].long()[place // page].cuda()
        keys[at, :, (place % page).cuda()], values[at, :, :, (place % page).cuda()] = k, v
        rows.append((k.double(), v.double()))
    return keys, values, table.cuda(), rows


def exact(q, rows, scale, window, softcap, chunk, slopes, sinks, gates):
    out = []
    for r, (k, v) in enumerate(rows):
        last, heads = k.shape[0] - 1, q.shape[1]
        place = torch.arange(last + 1, device="cuda")
        seen = torch.ones_like(place, dtype=torch.bool)
        if window:
            seen &= last - place < window
        if chunk:
            seen &= place // chunk == last // chunk
        for h in range(heads):
            kv = h // (heads // k.shape[1])
            s = k[:, kv] @ q[r, h].double() * scale
            s = softcap * torch.tanh(s / softcap) if softcap else s
            s = s - (float(slopes[h]) * (last - place) if slopes is not None else 0.0)
            s = s.masked_fill(~seen, -torch.inf)
            if sinks is not None:
                s = torch.cat([s, sinks[h:h + 1].double()])
            o = torch.softmax(s, dim=0)[:last + 1] @ v[:, kv]
            out.append(o * torch.sigmoid(gates[r, h].double()) if gates is not None else o)
    return torch.stack(out).view(len(rows), -1)


def staged_plan(contexts, group, n_kv, window=None, chunk=None):
    plan = build_attention_plan([1] * len(contexts), contexts, group, n_kv, window, merge_in_workgroup=4, chunk=chunk)
    to = lambda a: torch.from_numpy(a).cuda()
    return {"items": to(plan.items), "item_slot": to(plan.item_slot), "merges": to(plan.merges), "n_items": len(plan.items), "n_merges": 0,
            "n_slots": 0, "merge_in_workgroup": 4, "rows_in_order": True}


SHAPES = [(4, 2, 32, 16), (8, 8, 128, 16), (16, 8, 128, 32), (32, 8, 128, 16), (6, 2, 64, 48), (16, 1, 256, 16), (40, 2, 96, 16), (12, 1, 128, 64)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_q, n_kv, d, page", SHAPES)
@pytest.mark.parametrize("extra", ["plain", "window", "chunk", "softcap", "slopes", "sinks and gates"])
def test_one_token_a_row(ops, dtype, n_q, n_kv, d, page, extra):
    print(f"single tokens {dtype} {n_q}/{n_kv} d{d} page {page} {extra}", flush=True)
    assert ops._attention_library(dtype, d).lsa_attention_single_fits(page, 0)
    torch.manual_seed(n_q * d + page)
    rows = len(CONTEXTS)
    keys, values, table, exact_rows = pool(dtype, n_kv, d, page, CONTEXTS)
    qkv = torch.randn(rows, (n_q + 2 * n_kv) * d, device="cuda").to(dtype)
    window, chunk, softcap = 40 if extra == "window" else None, 48 if extra == "chunk" else None, 2.0 if extra == "softcap" else None
    slopes = torch.rand(n_q, device="cuda") * 0.1 if extra == "slopes" else None
    sinks = torch.randn(n_q, device="cuda") if "sinks" in extra else None
    gates = torch.randn(rows, n_q + 3, device="cuda").to(dtype)[:, 1:1 + n_q] if "gates" in extra else None
    if window:
        for r, c in enumerate(CONTEXTS):
            table[r, :max(0, c - window) // page] = -1                # pages that the window has passed are gone
    t = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    got = torch.full((rows, n_q * d), float("nan"), device="cuda", dtype=dtype)
    ops.paged_attention(qkv, got, keys, values, table, t(list(range(rows))), t([1] * rows), t(CONTEXTS), staged_plan(CONTEXTS, n_q // n_kv, n_kv, window, chunk),
                        d ** -0.5, window, page, n_q, n_kv, d, Ctx(), sinks=sinks, softcap=softcap, chunk=chunk, slopes=slopes, gates=gates)
    want = exact(qkv[:, :n_q * d].view(rows, n_q, d), exact_rows, d ** -0.5, window, softcap, chunk, slopes, sinks, gates)
    torch.testing.assert_close(got.double(), want, **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_q, n_kv, d, page", [shape for shape in SHAPES if shape[2] % 64 == 0])
@pytest.mark.parametrize("window", [None, 40])
def test_norm_rotation_and_cache_write(ops, dtype, n_q, n_kv, d, page, window):
    """The projection as it is: against the kernel that prepares it, and attention behind it; writing the cache, and reading one that is written."""
    print(f"single tokens fused {dtype} {n_q}/{n_kv} d{d} page {page} window {window}", flush=True)
    assert ops.single_token_fusion_fits(dtype, d, page)
    torch.manual_seed(n_q + d + page)
    rows = len(CONTEXTS)
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
    want = exact(ready[:, :n_q * d].view(rows, n_q, d), exact_rows, d ** -0.5, window, None, None, None, None, None)
    plan = staged_plan(CONTEXTS, n_q // n_kv, n_kv, window)
    for write, k, v in ((True, keys.clone(), values.clone()), (False, ready_k.clone(), ready_v.clone())):
        raw, got = qkv.clone(), torch.full((rows, n_q * d), float("nan"), device="cuda", dtype=dtype)
        ops.paged_attention(raw, got, k, v, table, order, t([1] * rows), t(CONTEXTS), plan, d ** -0.5, window, page, n_q, n_kv, d, Ctx(),
                            decode_fusion=(qw, kw, 1e-6, cos_sin, write))
        assert torch.equal(raw, qkv)
        torch.testing.assert_close(got.double(), want, **TOL[dtype])
        there = ~torch.isnan(ready_k)
        assert torch.equal(there, ~torch.isnan(k)) and torch.equal(torch.isnan(ready_v), torch.isnan(v)) and torch.equal(ready_v[~torch.isnan(v)], v[~torch.isnan(v)])
        torch.testing.assert_close(k[there].float(), ready_k[there].float(), **TOL[dtype])


def test_what_stays_with_the_other_kernels(ops):
    lib = ops._attention_library
    assert not lib(torch.bfloat16, 128).lsa_attention_single_fits(8, 0) and not lib(torch.bfloat16, 48).lsa_attention_single_fits(16, 0)
    assert not lib(torch.float32, 128).lsa_attention_single_fits(20, 0) and not lib(torch.float32, 48).lsa_attention_single_fits(16, 1)
    assert lib(torch.float32, 48).lsa_attention_single_fits(16, 0) and not lib(torch.bfloat16, 96).lsa_attention_single_fits(16, 1)
    assert np.all([lib(dtype, 128).lsa_attention_single_fits(page, 1) for dtype in (torch.float32, torch.bfloat16) for page in (16, 32, 48, 496)])
