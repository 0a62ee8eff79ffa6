"""Values of long steps whose tiles are shared by several workgroups (each takes some of a tile's dimensions): rows of one token, portions that meet in a tile, tiles
of fewer dimensions than a share, shares that end behind the values.  The same numbers as a few tokens at a time, which another kernel puts there; values are copies."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_q, n_kv, dim, value_dim, D", [(4, 1, 128, 128, 128), (2, 2, 8, 8, 16), (1, 1, 8, 8, 8), (2, 3, 40, 24, 48), (2, 40, 64, 64, 64), (1, 1, 120, 72, 120)])
@pytest.mark.parametrize("rows", [[(1, 3 * r) for r in range(260)], [(20, 5 * r) for r in range(14)], [(1, 17)] * 3 + [(700, 2)]])
def test_every_dimension_of_every_token(dtype, n_q, n_kv, dim, value_dim, D, rows):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    print(f"value parts {dtype} {n_q}/{n_kv} {dim} {value_dim} {D} {len(rows)} rows", flush=True)
    torch.manual_seed(dim + D)
    page = 16
    positions = torch.cat([torch.arange(b, b + c) for c, b in rows]).int().cuda()
    token_row = torch.cat([torch.full((c,), r) for r, (c, _) in enumerate(rows)]).int().cuda()
    width, tokens = max(-(-(c + b) // page) for c, b in rows), len(positions)
    table = torch.randperm(len(rows) * width).view(len(rows), width).int().cuda()
    qkv = torch.randn(tokens, (n_q + n_kv) * dim + n_kv * value_dim, device="cuda").to(dtype)
    weight, cos_sin = 1 + 0.2 * torch.randn(dim, device="cuda"), torch.randn(tokens, 8, device="cuda")
    results = []
    for step in (tokens, 64):
        keys, values = torch.full((len(rows) * width, n_kv, page, D), 3.0, device="cuda", dtype=dtype), torch.full((len(rows) * width, n_kv, D, page), 3.0, device="cuda", dtype=dtype)
        out = torch.full((tokens, n_q * D), float("nan"), device="cuda", dtype=dtype)
        for a in range(0, tokens, step):
            piece = slice(a, a + step)
            ops.qkv_prepare(qkv[piece], keys, values, table, token_row[piece], positions[piece], weight, weight, 1e-6, cos_sin[piece], page, n_q, n_kv, dim,
                            value_dim, out[piece])
        results.append((out, keys, values))
    assert torch.equal(results[0][2], results[1][2]) and not torch.isnan(results[0][0]).any()
    close = dict(rtol=2.0 ** -7, atol=2.0 ** -7) if dtype == torch.bfloat16 else dict(rtol=1e-5, atol=1e-5)        # (sums of squares in another order, then the rounding)
    torch.testing.assert_close(results[0][0], results[1][0], **close)
    torch.testing.assert_close(results[0][1], results[1][1], **close)
