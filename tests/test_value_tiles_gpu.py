"""Values of long steps, put into their pages by tiles of 64 tokens: portions that meet inside a tile at any place of a page, portions that go on
behind cached tokens, rows of one token among them, rows without a page.  A copy: every place holds the very number, no other place changes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d, page", [(16, 4), (128, 16), (96, 12), (256, 64)])
@pytest.mark.parametrize("rows", [[(300, 0)], [(97, 0), (1, 33), (1, 6), (131, 5), (70, 2), (3, 63)], [(1, i) for i in range(256)], [(255, 3), (1, 0)]])
def test_values_of_portions_that_meet_in_a_tile(dtype, d, page, rows):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    print(f"value tiles {dtype} d{d} page {page} {len(rows)} rows", flush=True)
    torch.manual_seed(d + page)
    n_q, n_kv = 2, 2
    positions = torch.cat([torch.arange(before, before + count) for count, before in rows]).int()
    token_row = torch.cat([torch.full((count,), r) for r, (count, _) in enumerate(rows)]).int()
    width = max(-(-(count + before) // page) for count, before in rows)
    pages = len(rows) * width + 2
    table = torch.randperm(pages)[:len(rows) * width].view(len(rows), width).int()
    if len(rows) > 2:
        table[2] = -1                                      # a row whose pages are not there writes nothing
    tokens = len(positions)
    qkv = torch.randn(tokens, (n_q + 2 * n_kv) * d, device="cuda").to(dtype)
    keys, values = torch.zeros(pages, n_kv, page, d, device="cuda", dtype=dtype), torch.full((pages, n_kv, d, page), 7.0, device="cuda", dtype=dtype)
    want = values.clone()
    for t in range(tokens):
        at = int(table[token_row[t], positions[t] // page])
        if at >= 0:
            want[at, :, :, int(positions[t]) % page] = qkv[t].view(-1, d)[n_q + n_kv:]
    ops.qk_norm_rope_kv_write(qkv, keys, values, table.cuda(), token_row.cuda(), positions.cuda(), None, None, 0.0, None, page, n_q, n_kv, d, True)
    assert torch.equal(values, want)
