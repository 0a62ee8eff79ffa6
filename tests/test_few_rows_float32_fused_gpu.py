"""What the 32-bit product for a few rows folds in, at the edges of its tiles: the row scale, the stream update, the gated activation, against 64 bits.

A product's error stays below K / 32 + 8 roundings of 2^-24 in the norm (32 chains); what is folded in adds a handful of roundings, and
silu a few more (expf is right to 2 units): 16 in all."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


def error(got, exact):
    return float((got.double() - exact).norm() / exact.norm())


def bound(inner):
    return (inner / 32 + 24) * 2.0 ** -24


def scaled_stream(generator, rows, inner, parts):
    """A stream times a norm's weights, partial sums of its squares, and the normalised rows in 64 bits."""
    stream = torch.randn(rows, inner, device="cuda", generator=generator)
    weight = 1 + 0.2 * torch.randn(inner, device="cuda", generator=generator)
    squares = torch.zeros(rows, parts, device="cuda", dtype=torch.float64)
    squares.index_add_(1, torch.arange(inner, device="cuda") % parts, stream.double() ** 2)
    normed = stream.double() * torch.rsqrt((stream.double() ** 2).mean(dim=1, keepdim=True) + 1e-6) * weight.double()
    return stream * weight, (squares.float(), 1e-6), normed


@pytest.mark.parametrize("rows, outputs, inner, parts", [(1, 1, 512, 1), (2, 4096, 1024, 128), (8, 1023, 580, 65), (3, 1024, 2048, 512), (5, 2050, 772, 300),
                                                         (7, 4100, 1024, 64)])
def test_row_scale_stream_and_gate(ops, rows, outputs, inner, parts):
    print(f"float32 few rows fused {rows} {outputs} {inner} {parts}", flush=True)
    generator = torch.Generator("cuda").manual_seed(rows + outputs)
    x, row_scale, normed = scaled_stream(generator, rows, inner, parts)
    w = torch.randn(outputs, inner, device="cuda", generator=generator)
    bias = torch.randn(outputs, device="cuda", generator=generator)
    exact = normed @ w.double().T
    assert error(ops._linear_few_rows_float32(x, w, None, bias, row_scale), exact + bias.double()) < bound(inner)
    if ops.row_scale_fits(x, w, row_scale):
        assert error(ops.linear_few_rows(x, w, row_scale=row_scale), exact) < bound(inner)
        resid, norm_weight = torch.randn(rows, outputs, device="cuda", generator=generator), 1 + 0.2 * torch.randn(outputs, device="cuda", generator=generator)
        kept = resid.clone()
        for scale, update in ((row_scale, exact), (None, x.double() @ w.double().T)):
            stream, weighted, squares = ops.linear_into_stream(x, w, resid, norm_weight, row_scale=scale)
            want = resid.double() + update
            assert torch.equal(resid, kept) and error(stream, want) < bound(inner)
            assert torch.equal(weighted, stream * norm_weight)
            assert error(squares.sum(dim=1), (stream.double() ** 2).sum(dim=1)) < 16 * 2.0 ** -24
            assert squares.shape[1] <= ops.SCALE_PARTS


@pytest.mark.parametrize("rows, pairs, inner, parts", [(1, 1, 512, 1), (2, 3072, 1024, 128), (8, 513, 1024, 40), (6, 1023, 2048, 256), (4, 2049, 900, 7)])
def test_gated(ops, rows, pairs, inner, parts):
    print(f"float32 few rows gated {rows} {pairs} {inner} {parts}", flush=True)
    generator = torch.Generator("cuda").manual_seed(rows + pairs)
    x, row_scale, normed = scaled_stream(generator, rows, inner, parts)
    w = torch.randn(2 * pairs, inner, device="cuda", generator=generator) * inner ** -0.5
    for scale, rows_of in ((row_scale, normed), (None, x.double())):
        got = ops.linear_gated(x, w, row_scale=scale)
        if not ops._fuses_float32(x, w, scale):
            assert got is None
            continue
        gate, up = (rows_of @ w.double().T).chunk(2, dim=1)
        assert error(got, gate * torch.sigmoid(gate) * up) < 2 * bound(inner)          # (two products meet)


def test_what_is_not_folded_in(ops):
    make = lambda *shape: torch.randn(*shape, device="cuda")
    sums = lambda rows, parts: (torch.ones(rows, parts, device="cuda"), 1e-6)
    w, resid, weight = make(1024, 1024), make(9, 1024), make(1024)
    assert ops.linear_into_stream(make(9, 1024), w, resid, weight) is None and ops.linear_gated(make(9, 1024), w) is None
    assert not ops.row_scale_fits(make(9, 1024), w, sums(9, 8)) and not ops.row_scale_fits(make(2, 1024), w, sums(2, 513))
    assert ops.linear_into_stream(make(2, 1024), w, make(2, 1024).bfloat16(), weight) is None
    assert ops.linear_gated(make(2, 1024), w, activation="gelu_tanh") is None and ops.linear_few_rows(make(2, 1024), w) is None
