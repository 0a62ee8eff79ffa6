"""The sorted products of routed experts at the sizes where their tiles can go wrong, against every pair on its own in float32.

A pair's hidden row is a float32 sum rounded to bfloat16 on either side, so an output is off by a share of bfloat16's step of
the hidden row (2^-9 of its numbers, as many as there are, no two alike): 2^-9 of the output's norm bounds it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


# (experts, pairs of each of the first experts, the others have none; width, inter, with gates); the wide tiles begin at 40 pairs an expert
@pytest.mark.parametrize("experts,counts,width,inter,gated", [
    (1, [40], 32, 32, True), (1, [256], 64, 128, False), (2, [257, 1], 96, 160, True), (3, [64, 65, 600], 128, 96, False),
    (9, [40] * 9, 64, 288, True), (5, [0, 511, 0, 513, 255], 192, 64, False), (20, [2500] + [0] * 18 + [3], 64, 32, True),
    (4, [15, 16, 17, 80], 64, 64, True), (33, [1] * 33, 32, 64, False), (33, [1] * 32, 32, 64, False), (33, [1] * 32 + [2], 32, 64, False), (70, [7] * 70, 96, 32, True)])
def test_sorted_products_at_the_edges_of_their_tiles(ops, experts, counts, width, inter, gated):
    print(f"expert tiles {experts} {counts[:5]} {width} {inter} {gated}", flush=True)
    generator = torch.Generator("cuda").manual_seed(width + inter)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    owner = torch.cat([torch.full((count,), e, dtype=torch.int32) for e, count in enumerate(counts)])
    owner = owner[torch.randperm(len(owner), generator=torch.Generator().manual_seed(1))].cuda()
    n = len(owner)
    chosen, weights = owner.view(n, 1).contiguous(), draw(n, 1)
    x = draw(n, width).to(torch.bfloat16)
    up = (draw(experts, (2 if gated else 1) * inter, width) / width ** 0.5).to(torch.bfloat16)
    down = (draw(experts, width, inter) / inter ** 0.5).to(torch.bfloat16)
    out = torch.full((n, width), float("nan"), device="cuda")
    taken = ops.experts_sorted(x, up, down, chosen, weights, out, **({} if gated else {"activation": "relu2"}))
    assert taken == (n > experts)
    if not taken:
        return
    want = torch.empty_like(out)
    for e in range(experts):
        rows = (owner == e).nonzero().flatten()
        y = x[rows].float() @ up[e].float().T
        y = torch.nn.functional.silu(y[:, :inter]) * y[:, inter:] if gated else y.clamp(min=0) ** 2
        want[rows] = weights[rows] * (y.to(torch.bfloat16).float() @ down[e].float().T)
    forms = []
    for tile_rows in (64, 256):                                # (whichever the sizes ask for)
        forms.append(torch.full((n, width), float("nan"), device="cuda"))
        assert ops.experts_sorted(x, up, down, chosen, weights, forms[-1], tile_rows=tile_rows, **({} if gated else {"activation": "relu2"}))
    assert torch.equal(forms[0], forms[1]) and (torch.equal(out, forms[0]))       # (both add a sum's products in the same order)
    assert torch.isfinite(out).all()
    assert float((out - want).norm() / want.norm()) < 2.0 ** -9
    assert float(((out - want).norm(dim=1) / want.norm(dim=1)).max()) < 2.0 ** -7


# (experts, choices a token, tokens, width, inter): the wide tiles at models' sizes, 48 and 75 pairs an expert; 16.5 slabs of 64 in the second product
@pytest.mark.parametrize("activation,limit", [("silu", 0.0), ("clamped", 0.7), ("relu2", 0.0)])
@pytest.mark.parametrize("experts,top,n,width,inter", [(64, 6, 512, 2048, 1408), (16, 4, 300, 4096, 1056)])
def test_sorted_products_at_models_sizes(ops, experts, top, n, width, inter, activation, limit):
    """Experts that have nothing in common and are chosen unevenly, some of them by nobody: a pair at another expert or a slip in a slab shows in its
    token's row.  If every number of a hidden row were rounded the other way, the row would be off by 2^-8."""
    print(f"expert tiles at models' sizes {experts} {top} {n} {width} {inter} {activation}", flush=True)
    generator = torch.Generator("cuda").manual_seed(inter)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    wanted = draw(experts).exp()
    wanted[::7] = 0                                            # (nobody's)
    chosen = torch.multinomial(wanted.expand(n, -1), top, generator=generator).to(torch.int32)
    weights, x = draw(n, top), draw(n, width).to(torch.bfloat16)
    up = (draw(experts, (1 if activation == "relu2" else 2) * inter, width) / width ** 0.5).to(torch.bfloat16)
    down = (draw(experts, width, inter) / inter ** 0.5).to(torch.bfloat16)
    lib = ops._part_library("experts")
    assert lib.lsa_experts_tile_rows(n * top, experts, inter, width, int(activation == "relu2"), 1) == 256
    more = {} if activation == "silu" else {"activation": activation, "limit": limit} if limit else {"activation": activation}
    outs = {}
    for tile_rows in (0, 64, 256):
        outs[tile_rows] = torch.full((n, width), float("nan"), device="cuda")
        assert ops.experts_sorted(x, up, down, chosen, weights, outs[tile_rows], tile_rows=tile_rows, **more)
    assert torch.equal(outs[0], outs[256]) and torch.equal(outs[64], outs[256])
    want = torch.zeros(n, width, device="cuda")
    for e in range(experts):
        rows, places = (chosen == e).nonzero(as_tuple=True)
        y = x[rows].float() @ up[e].float().T
        gate, rest = y[:, :inter], y[:, inter:]
        if activation == "silu":
            y = torch.nn.functional.silu(gate) * rest
        elif activation == "clamped":
            gate = gate.clamp(max=limit)
            y = gate * torch.sigmoid(1.702 * gate) * (rest.clamp(-limit, limit) + 1.0)
        else:
            y = y.clamp(min=0) ** 2
        want.index_add_(0, rows, weights[rows, places, None] * (y.to(torch.bfloat16).float() @ down[e].float().T))
    off = (outs[0] - want).norm(dim=1) / want.norm(dim=1)
    print("off a token", float(off.max()), flush=True)
    assert float(off.max()) < 2.0 ** -8
