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
