"""Kernels over rows of a 32-bit stream at widths on both sides of every piece that a thread may take (one or four columns, 256 or 1,024 threads, rows
longer than registers keep), at addresses that are and are not multiples of 16 bytes, against 64 bits.

Sums of `width` squares in float32, at most 64 a thread and ten across: 2e-6 relative; bfloat16 results are rounded once more (2^-9)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
WIDTHS = [4, 6, 100, 1028, 2052, 4099, 4100, 8200]


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


def near(got, want):
    torch.testing.assert_close(got.double(), want, **(dict(rtol=2.0 ** -8, atol=1e-3) if got.dtype == torch.bfloat16 else dict(rtol=5e-6, atol=5e-6)))


def shifted(*shape, offset=0, dtype=torch.float32):
    count = 1
    for size in shape:
        count *= size
    return torch.randn(count + offset, device="cuda").to(dtype)[offset:].view(*shape)


def unit(x, eps=1e-6):
    return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + eps)


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_norm_of_chosen_rows_and_of_embeddings(ops, width, offset, out_dtype):
    print(f"norm rows {width} {offset} {out_dtype}", flush=True)
    torch.manual_seed(width)
    x, weight = shifted(5, width, offset=offset), torch.randn(width, device="cuda")
    rows = torch.tensor([4, 0, 4], device="cuda", dtype=torch.int32)
    for chosen, index in ((None, slice(None)), (rows, rows.long())):
        out = torch.full((5 if chosen is None else 3, width), float("nan"), device="cuda", dtype=out_dtype)
        ops.norm_rows(x, chosen, weight, 1e-6, out)
        near(out, unit(x[index].double()) * weight.double())
    table, out = shifted(7, width, offset=offset, dtype=out_dtype), torch.full((4, width), float("nan"), device="cuda")
    ids = torch.tensor([6, 0, 9, -1], device="cuda", dtype=torch.int32)                # (ids outside the table give rows of zeros)
    ops.embedding_norm(table, ids, weight, 1e-6, out)
    near(out[:2], unit(table[ids[:2].long()].double()) * weight.double())
    assert not out[2:].any()


@pytest.mark.parametrize("width", [4, 6, 1028, 2052])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("offset", [0, 1])
def test_short_convolution(ops, width, taps, offset):
    """Tokens of portions that begin a sequence, go on behind one or many tokens, and single tokens whose state moves on in the same launch."""
    print(f"short conv {width} {taps} {offset}", flush=True)
    torch.manual_seed(width + taps)
    for rows in ([(5, 0), (1, 0), (3, 1), (2, 9)], [(1, 0), (1, 1), (1, 2), (1, 7)]):
        keep = int(all(count == 1 for count, _ in rows))
        tokens = sum(count for count, _ in rows)
        x, w, state = shifted(tokens, width, offset=offset), torch.randn(width, taps, device="cuda"), torch.randn(len(rows), max(taps - 1, 1), width, device="cuda")
        old = state.clone()
        slots = torch.randperm(len(rows)).int().cuda()
        start = torch.tensor([sum(c for c, _ in rows[:r]) for r in range(len(rows))], dtype=torch.int32, device="cuda")
        token_row = torch.cat([torch.full((c,), r) for r, (c, _) in enumerate(rows)]).int().cuda()
        positions = torch.cat([torch.arange(b, b + c) for c, b in rows]).int().cuda()
        out = torch.full((tokens, width), float("nan"), device="cuda")
        ops.short_conv(x, w, state, slots, token_row, positions, start, out, keep=bool(keep))
        want = x.double().clone()
        for t in range(tokens):
            r, position = int(token_row[t]), int(positions[t])
            first = position - (t - int(start[r]))
            for j in range(taps):
                place = position - (taps - 1 - j)
                if place >= first:
                    want[t] += w[:, j].double() * x[t - (position - place)].double()
                elif place >= 0:
                    want[t] += w[:, j].double() * old[int(slots[r]), taps - 1 - (first - place)].double()
        near(out, want)
        if keep and taps > 1:
            for r in range(len(rows)):
                assert torch.equal(state[int(slots[r])], torch.cat([old[int(slots[r]), 1:], x[r:r + 1]]))
        else:
            assert torch.equal(state, old)


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("streams, rows", [(1, 3), (2, 300), (3, 1), (8, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_streams_read_and_update(ops, width, streams, rows, dtype):
    print(f"streams {width} {streams} {rows} {dtype}", flush=True)
    torch.manual_seed(width + streams)
    x, y = torch.randn(streams, rows, width, device="cuda"), shifted(rows, width, offset=width % 3, dtype=dtype)
    read, mix, write, weight = torch.randn(streams, device="cuda"), torch.randn(streams, streams, device="cuda"), torch.randn(streams, device="cuda"), torch.randn(width, device="cuda")
    out = torch.full((rows, width), float("nan"), device="cuda", dtype=dtype)
    ops.streams_read(x, read, weight, 1e-6, out)
    near(out, unit(torch.einsum("s,stw->tw", read.double(), x.double())) * weight.double())
    fresh = torch.einsum("st,snw->tnw", mix.double(), x.double()) + write.double()[:, None, None] * y.double()
    for normed in (False, True):
        again, out = x.clone(), torch.full((rows, width), float("nan"), device="cuda", dtype=dtype)
        ops.streams_update(again, y, mix, write, *((read, weight, 1e-6, out) if normed else ()))
        near(again, fresh)
        if normed:
            near(out, unit(torch.einsum("s,stw->tw", read.double(), fresh)) * weight.double())


@pytest.mark.parametrize("width", [4, 6, 1028, 4100, 8200])
@pytest.mark.parametrize("before", [None, 0, 3])
@pytest.mark.parametrize("offset", [0, 1])
def test_scaled_norm_and_sum(ops, width, before, offset):
    print(f"scaled norm add {width} {before} {offset}", flush=True)
    torch.manual_seed(width)
    x, y = shifted(3, width, offset=offset), shifted(3, width, offset=offset, dtype=torch.bfloat16)
    weight, scale = torch.randn(width, device="cuda"), torch.randn(width, device="cuda")
    out, rounded = torch.full((3, width), float("nan"), device="cuda"), torch.full((3, width), float("nan"), device="cuda", dtype=torch.bfloat16)
    summed = x.double() + unit(y.double()) * weight.double() * scale.double()
    after, want = {}, summed
    if before is not None:
        history, mix = torch.randn(before + 2, 3, width, device="cuda"), torch.randn(before + 1, device="cuda")
        want = torch.einsum("j,jtw->tw", mix[:before].double(), history[:before].double()) + mix[before].double() * summed
        after = {"history": history, "before": before, "mix": mix}
    ops.scaled_norm_add(x, y, weight, scale, 1e-6, out, rounded=rounded, **after)
    near(out, want)
    near(rounded, want)
    if before is not None:
        near(history[before], summed)
