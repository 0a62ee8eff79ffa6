"""Kernels that take several neighbouring columns a thread where widths and addresses allow it, at widths and addresses on both sides, against
what they compute written out in torch (the same roundings: equal numbers)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows, width, offset", [([(3, 0), (1, 5)], 40, 0), ([(200, 0), (130, 7), (1, 0), (2, 3)], 1000, 0), ([(130, 2), (140, 0)], 1004, 0),
                                                 ([(260, 0), (9, 1)], 1024, 0), ([(260, 1)], 1024, 1), ([(4, 0)] * 70, 2056, 0)])
def test_token_shift(ops, dtype, rows, width, offset):
    print(f"token shift {dtype} {len(rows)} rows {width} {offset}", flush=True)
    torch.manual_seed(width + offset)
    tokens = sum(count for count, _ in rows)
    h = torch.randn(tokens * width + offset, device="cuda").to(dtype)[offset:].view(tokens, width)
    mu, state = torch.rand(3, width, device="cuda"), torch.randn(len(rows) + 1, width, device="cuda")
    slots = torch.randperm(len(rows) + 1)[:len(rows)].int().cuda()
    start = torch.tensor([sum(c for c, _ in rows[:r]) for r in range(len(rows))], dtype=torch.int32, device="cuda")
    token_row = torch.cat([torch.full((c,), r) for r, (c, _) in enumerate(rows)]).int().cuda()
    positions = torch.cat([torch.arange(b, b + c) for c, b in rows]).int().cuda()
    out = torch.full((3, tokens, width), float("nan"), device="cuda", dtype=dtype)
    lib = ops._part_library("recurrent")
    assert lib.lsa_token_shift(0 if dtype == torch.float32 else 1, h.data_ptr(), mu.data_ptr(), 3, state.data_ptr(), state.stride(0), slots.data_ptr(), token_row.data_ptr(),
                               positions.data_ptr(), start.data_ptr(), out.data_ptr(), tokens, width, 0, torch.cuda.current_stream().cuda_stream) == 0
    own = h.double()
    before = torch.cat([torch.zeros_like(own[:1]), own[:-1]])
    first = (torch.arange(tokens, device="cuda") == start[token_row.long()].long())
    before[first] = state[slots.long()[token_row.long()[first]]].double()
    before[positions == 0] = 0.0
    want = own + (before - own) * mu.double()[:, None]
    torch.testing.assert_close(out.double(), want, rtol=2.0 ** -7 if dtype == torch.bfloat16 else 1e-6, atol=1e-6 if dtype == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens, heads, dim, rot, rank, row, offset", [(20, 5, 24, 16, 40, 64, 0), (33, 4, 16, 8, 30, 48, 0), (18, 9, 128, 64, 192, 256, 0),
                                                                        (17, 1, 8, 4, 6, 16, 0), (40, 6, 32, 32, 100, 144, 2), (24, 16, 64, 64, 512, 592, 0)])
def test_query_rows_of_a_latent(ops, dtype, tokens, heads, dim, rot, rank, row, offset):
    """Query rows put together from what a product left: the latent part is a copy, the rotated part within roundings, zeros behind it."""
    print(f"latent rows {dtype} {tokens} {heads} {rank} {row} {offset}", flush=True)
    torch.manual_seed(rank + row)
    stride = heads * (dim + rot) + rank + rot
    proj = torch.randn(tokens, stride, device="cuda").to(dtype)
    latent = torch.randn(heads * tokens * rank + offset, device="cuda").to(dtype)[offset:].view(heads, tokens, rank)
    cs = torch.randn(tokens, rot, device="cuda")
    norm = torch.ones(rank, device="cuda")
    page = 16
    keys, values = torch.zeros(tokens // page + 2, page, row, device="cuda", dtype=dtype), torch.zeros(tokens // page + 2, row, page, device="cuda", dtype=dtype)
    table = torch.arange(tokens // page + 2, device="cuda", dtype=torch.int32)[None].contiguous()
    zero, positions = torch.zeros(tokens, device="cuda", dtype=torch.int32), torch.arange(tokens, device="cuda", dtype=torch.int32)
    out = torch.full((tokens, heads, row), float("nan"), device="cuda", dtype=dtype)
    lib, p = ops._part_library("latent"), lambda tensor: tensor.data_ptr()
    assert lib.lsa_latent_prepare(0 if dtype == torch.float32 else 1, p(proj), stride, p(latent), None, p(norm), 1e-6, p(cs), rot // 2, p(keys), p(values), p(table),
                                  table.shape[1], p(zero), p(positions), page, p(out), heads, dim, rot, rank, row, 1, tokens, 0, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out[..., :rank], latent.transpose(0, 1)) and not out[..., rank + rot:].any()
    turned = proj[:, :heads * (dim + rot)].view(tokens, heads, dim + rot)[..., dim:].double()
    c, s = cs.double()[:, None, :rot // 2], cs.double()[:, None, rot // 2:]
    u, v = turned[..., 0::2], turned[..., 1::2]
    want = torch.stack([u * c - v * s, v * c + u * s], dim=-1).flatten(-2)
    torch.testing.assert_close(out[..., rank:rank + rot].double(), want, rtol=2.0 ** -8 if dtype == torch.bfloat16 else 1e-5, atol=2.0 ** -8 if dtype == torch.bfloat16 else 1e-5)
    assert keys.any() and torch.equal(keys, values.transpose(1, 2))


CLOSE = {torch.float32: dict(rtol=1e-5, atol=1e-5), torch.bfloat16: dict(rtol=2.0 ** -7, atol=2.0 ** -7)}      # (sums of squares in another order, then the rounding)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_q, n_kv, dim, value_dim, D, pairs, pairing, share, norm, write", [
    (4, 2, 128, 128, 128, 32, "neighbours", 1, True, True), (3, 1, 40, 24, 48, 16, "halves", 1, True, True), (16, 16, 128, 128, 128, 0, "halves", 2, False, True),
    (2, 2, 64, 64, 64, 32, "halves", 1, True, False), (1, 1, 8, 16, 16, 4, "neighbours", 1, True, True), (5, 5, 96, 96, 96, 20, "neighbours", 1, False, True)])
def test_long_preparation_of_queries_keys_and_values(ops, dtype, n_q, n_kv, dim, value_dim, D, pairs, pairing, share, norm, write):
    """All tokens of three portions at once, against the same tokens a few at a time, which another kernel prepares."""
    print(f"qkv prepare long {dtype} {n_q}/{n_kv} {dim} {value_dim} {D} {pairs} {pairing} {share}", flush=True)
    torch.manual_seed(dim + D)
    page, rows = 16, [(203, 0), (1, 40), (97, 5)]
    tokens = sum(count for count, _ in rows)
    positions = torch.cat([torch.arange(b, b + c) for c, b in rows]).int().cuda()
    token_row = torch.cat([torch.full((c,), r) for r, (c, _) in enumerate(rows)]).int().cuda()
    width = 16
    table = torch.randperm(3 * width).view(3, width).int().cuda()
    stride = -(-(n_q + n_kv) * dim // 8) * 8 + -(-(n_kv // share) * value_dim // 8) * 8 + 8
    qkv = torch.randn(tokens, stride, device="cuda").to(dtype)
    weights = [1 + 0.2 * torch.randn(dim, device="cuda") if norm else None for _ in range(2)]
    cs = torch.randn(tokens, 2 * pairs, device="cuda") if pairs else None
    def run(pieces):
        keys, values = torch.full((3 * width, n_kv, page, D), 3.0, device="cuda", dtype=dtype), torch.full((3 * width, n_kv, D, page), 3.0, device="cuda", dtype=dtype)
        out = torch.full((tokens, n_q * D), float("nan"), device="cuda", dtype=dtype)
        lib, p = ops._rope_kv, lambda tensor: None if tensor is None else tensor.data_ptr()
        for a, b in pieces:
            assert lib.lsa_qkv_prepare(0 if dtype == torch.float32 else 1, p(qkv[a:b]), stride, p(keys), p(values), p(table), width, p(token_row[a:b]), p(positions[a:b]),
                                       p(weights[0]), p(weights[1]), 1e-6, p(cs[a:b]) if cs is not None else None, pairs, page, n_q, n_kv, dim, value_dim, D, p(out[a:b]),
                                       1 if write else 0, b - a, 1 if pairing == "halves" else 0, share, torch.cuda.current_stream().cuda_stream) == 0
        return out, keys, values
    got, want = run([(0, tokens)]), run([(a, min(a + 100, tokens)) for a in range(0, tokens, 100)])
    torch.testing.assert_close(got[0], want[0], **CLOSE[dtype])
    torch.testing.assert_close(got[1], want[1], **CLOSE[dtype])
    assert torch.equal(got[2], want[2]) and not torch.isnan(got[0]).any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens, heads, value_dim, per_channel, kind, below", [(300, 16, 128, 0, 0, False), (1100, 4, 256, 1, 1, True), (4097, 1, 8, 1, 1, False),
                                                                                (600, 7, 136, 0, 1, True), (512, 8, 64, 1, 0, False)])
def test_long_norm_and_gate_of_heads(ops, dtype, tokens, heads, value_dim, per_channel, kind, below):
    print(f"norm and gate long {dtype} {tokens} {heads} {value_dim}", flush=True)
    torch.manual_seed(tokens + heads)
    x, weight = torch.randn(tokens, heads, value_dim, device="cuda"), torch.randn(heads if per_channel else 1, value_dim, device="cuda")
    gate_stride = heads * value_dim + 16
    gate = torch.randn(tokens, gate_stride, device="cuda").to(dtype)
    under = torch.rand(tokens, heads, 2, device="cuda") if below else None
    out = torch.full((tokens, heads * value_dim), float("nan"), device="cuda", dtype=dtype)
    lib, p = ops._part_library("recurrent"), lambda tensor: None if tensor is None else tensor.data_ptr()
    def run(out, a, b):
        assert lib.lsa_heads_norm_gate(0 if dtype == torch.float32 else 1, p(x[a:b]), p(weight), per_channel, 1e-6, p(gate[a:b]), gate_stride, p(out[a:b]), b - a, heads, value_dim,
                                       kind, p(under[a:b]) if below else None, 1e-6, torch.cuda.current_stream().cuda_stream) == 0
    run(out, 0, tokens)
    wide = x.double() / (torch.maximum(under[..., 0].abs(), under[..., 1])[..., None].double() + 1e-6 if below else 1.0)
    g = gate[:, :heads * value_dim].double().view(tokens, heads, value_dim)
    want = wide * torch.rsqrt(wide.pow(2).mean(dim=-1, keepdim=True) + 1e-6) * weight.double() * (torch.sigmoid(g) if kind else g * torch.sigmoid(g))
    torch.testing.assert_close(out.double().view_as(want), want, **CLOSE[dtype])
    eights, whole = out, gate
    out, gate = torch.full_like(out, float("nan")), torch.cat([whole.flatten()[:1], whole.flatten()])[1:].view_as(whole)      # the same gates at an odd address: the other form takes them
    run(out, 0, tokens)
    torch.testing.assert_close(eights, out, **CLOSE[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kv_heads, heads, dim, value_dim, taps, per_channel", [(2, 4, 128, 128, 4, 0), (1, 1, 8, 16, 2, 1), (3, 3, 40, 24, 3, 1), (2, 2, 64, 128, 4, 1)])
@pytest.mark.parametrize("rows", [[(1, 0), (1, 1), (1, 2), (1, 3), (1, 50)], [(70, 0), (1, 2), (2, 1), (5, 7)]])
def test_inputs_of_the_delta_rule(ops, dtype, kv_heads, heads, dim, value_dim, taps, per_channel, rows):
    """Rows at multiples of 16 bytes against the same rows elsewhere, which another kernel takes: read-outs, decays, strengths and the state."""
    print(f"delta inputs {dtype} {kv_heads} {heads} {dim} {value_dim} {taps} {per_channel} {len(rows)}", flush=True)
    torch.manual_seed(dim + taps)
    tokens, keep = sum(c for c, _ in rows), int(all(c == 1 for c, _ in rows))
    channels = 2 * kv_heads * dim + heads * value_dim
    stride = -(-(channels + 2 * heads) // 8) * 8
    numbers = torch.randn(tokens * stride, device="cuda").to(dtype)
    w, old = torch.randn(channels, taps, device="cuda"), torch.randn(len(rows), (taps - 1) * channels + 4, device="cuda")
    slots = torch.randperm(len(rows)).int().cuda()
    start = torch.tensor([sum(c for c, _ in rows[:r]) for r in range(len(rows))], dtype=torch.int32, device="cuda")
    token_row = torch.cat([torch.full((c,), r) for r, (c, _) in enumerate(rows)]).int().cuda()
    positions = torch.cat([torch.arange(b, b + c) for c, b in rows]).int().cuda()
    wide = heads * dim if per_channel else heads
    z = torch.randn(tokens, wide, device="cuda")
    scale, bias = torch.randn(heads, device="cuda"), torch.randn(wide, device="cuda")
    lib, p = ops._part_library("delta"), lambda tensor: tensor.data_ptr()
    def run(offset):
        proj = torch.cat([numbers.new_zeros(offset), numbers])[offset:].view(tokens, stride)
        state, out = old.clone(), torch.full((tokens, channels), float("nan"), device="cuda")
        strengths, decays = torch.full((tokens, heads), float("nan"), device="cuda"), torch.full((tokens, wide), float("nan"), device="cuda")
        strength = proj[:, channels:]
        decay = z if per_channel else proj[:, channels + heads:]
        assert lib.lsa_delta_prepare(0 if dtype == torch.float32 else 1, p(proj), stride, p(w), taps, p(state), state.stride(0), p(slots), p(token_row), p(positions), p(start),
                                     p(out), kv_heads, heads, dim, value_dim, dim ** -0.5, 1e-6, keep, p(strength), stride, p(decay), wide if per_channel else stride,
                                     per_channel, p(scale), p(bias), p(strengths), p(decays), tokens, torch.cuda.current_stream().cuda_stream) == 0
        return out, strengths, decays, state
    got, want = run(0), run(1)
    torch.testing.assert_close(got[0], want[0], rtol=1e-5, atol=1e-5)
    assert all(torch.equal(a, b) for a, b in zip(got[1:], want[1:])) and not torch.isnan(got[0]).any()
    assert keep or torch.equal(got[3], old)
