"""The tiles of 256 x 256 whose wavefronts take turns (``csrc/wide_product.hpp``) at the edges of what they leave out: blocks of 64 rows that are padding, columns from
128 on that the matrix does not have, slabs of 64 and a half one, from a single half slab on.

The narrow tiles add a sum's products in the same order, so the two agree bit by bit.  Against the products in 64 bits, whose hidden rows are rounded to bfloat16 as well: where sums in 32
and in 64 bits lie on two sides of a rounding's edge a hidden number is off by up to 2^-8 of it; few are, and the limit for the norm, 2^-9, is what was observed with room, not a bound."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,inter,gated", [(32, 64, True), (64, 32, False), (96, 128, True), (128, 160, False), (160, 288, True), (192, 384, False), (320, 224, True)])
@pytest.mark.parametrize("counts", [[1, 63, 64, 65], [127, 128, 129, 300], [191, 192, 193, 0], [255, 256, 257, 512]])
def test_blocks_of_rows_and_columns_that_are_left_out(counts, width, inter, gated):
    from llmserver_amd.kernels import default_ops
    print(f"wide products {counts} {width} {inter} {gated}", flush=True)
    ops, experts = default_ops(), len(counts)
    generator = torch.Generator("cuda").manual_seed(sum(counts) + width)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    owner = torch.cat([torch.full((count,), e, dtype=torch.int32) for e, count in enumerate(counts)])
    owner = owner[torch.randperm(len(owner), generator=torch.Generator().manual_seed(3))].cuda()
    n = len(owner)
    weights, x = draw(n, 1), draw(n, width).to(torch.bfloat16)
    up = (draw(experts, (2 if gated else 1) * inter, width) / width ** 0.5).to(torch.bfloat16)
    down = (draw(experts, width, inter) / inter ** 0.5).to(torch.bfloat16)
    outs = []
    for tile_rows in (64, 256):
        outs.append(torch.full((n, width), float("nan"), device="cuda"))
        assert ops.experts_sorted(x, up, down, owner.view(n, 1).contiguous(), weights, outs[-1], tile_rows=tile_rows, **({} if gated else {"activation": "relu2"}))
    assert torch.equal(outs[0], outs[1])
    want = torch.zeros(n, width, device="cuda", dtype=torch.float64)
    for e in range(experts):
        rows = (owner == e).nonzero().flatten()
        y = x[rows].double() @ up[e].double().T
        y = torch.nn.functional.silu(y[:, :inter]) * y[:, inter:] if gated else y.clamp(min=0) ** 2
        want[rows] = weights[rows].double() * (y.to(torch.bfloat16).double() @ down[e].double().T)
    assert float((outs[1] - want).norm() / want.norm()) < 2.0 ** -9
