"""Few pairs an expert: tiles of 64 pairs whose slabs go through LDS without registers, against the tiles that they stand beside (which take what does not begin at multiples
of 16 bytes) and against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def at_an_odd_place(tensor):
    return torch.empty(tensor.numel() + 1, device=tensor.device, dtype=tensor.dtype)[1:].view(tensor.shape).copy_(tensor)


# Pairs of each expert around the edges of 16, 32 and 64 rows; columns that end inside a block of 64 or 128; from one slab to more than there are buffers for.
@pytest.mark.parametrize("width,inter,activation,limit", [(64, 64, "silu", 0.0), (128, 160, "relu2", 0.0), (192, 128, "clamped", 0.7), (256, 320, "silu", 0.0), (448, 96, "relu2", 0.0),
                                                          (512, 704, "silu", 0.0)])
@pytest.mark.parametrize("counts", [[1, 2, 15, 16, 17], [31, 32, 33, 0, 48], [63, 64, 65, 0, 1], [129, 0, 0, 0, 191], [5] * 5])
def test_blocks_of_pairs_and_columns_at_their_edges(counts, width, inter, activation, limit):
    from llmserver_amd.kernels import default_ops
    print(f"expert streams {counts} {width} {inter} {activation}", flush=True)
    ops, experts = default_ops(), len(counts)
    generator = torch.Generator("cuda").manual_seed(sum(counts) + width)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    owner = torch.cat([torch.full((count,), e, dtype=torch.int32) for e, count in enumerate(counts)])
    owner = owner[torch.randperm(len(owner), generator=torch.Generator().manual_seed(3))].cuda().view(-1, 1).contiguous()
    n, plain = len(owner), activation == "relu2"
    weights, x = draw(n, 1), draw(n, width).to(torch.bfloat16)
    up = (draw(experts, (1 if plain else 2) * inter, width) / width ** 0.5).to(torch.bfloat16)
    down = (draw(experts, width, inter) / inter ** 0.5).to(torch.bfloat16)
    more = {"activation": activation, **({"limit": limit} if limit else {})}
    out, beside = (torch.full((n, width), float("nan"), device="cuda") for _ in range(2))
    assert ops.experts_sorted(x, up, down, owner, weights, out, tile_rows=64, **more)
    assert ops.experts_sorted(at_an_odd_place(x), at_an_odd_place(up), at_an_odd_place(down), owner, weights, beside, tile_rows=64, **more)
    assert torch.equal(out, beside)                            # (both add a sum's products in the same order)
    want = torch.zeros(n, width, device="cuda", dtype=torch.float64)
    for e in range(experts):
        rows = (owner.flatten() == e).nonzero().flatten()
        y = x[rows].double() @ up[e].double().T
        gate, rest = y[:, :inter], y[:, inter:]
        if plain:
            y = y.clamp(min=0) ** 2
        elif limit:
            gate = gate.clamp(max=limit)
            y = gate * torch.sigmoid(1.702 * gate) * (rest.clamp(-limit, limit) + 1.0)
        else:
            y = torch.nn.functional.silu(gate) * rest
        want[rows] = weights[rows].double() * (y.to(torch.bfloat16).double() @ down[e].double().T)
    assert float((out - want).norm() / want.norm()) < 2.0 ** -8      # (a hidden row is rounded to bfloat16 once, up to 2^-8 of each number)


def test_steps_of_models_sizes_choose_either_tiles():
    """32 tokens of 6 among 64 experts (the streams) and of 4 among 32 larger ones (12 tokens: the others for the first product), unevenly chosen, against the wide
    tiles bit by bit."""
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    for experts, top, n, width, inter in ((64, 6, 32, 2048, 1408), (32, 4, 12, 4096, 2048), (8, 2, 40, 2048, 1408)):
        print(f"expert streams at models' sizes {experts} {top} {n}", flush=True)
        generator = torch.Generator("cuda").manual_seed(inter)
        draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
        chosen = torch.multinomial(draw(experts).exp().expand(n, -1), top, generator=generator).to(torch.int32)
        weights, x = draw(n, top), draw(n, width).to(torch.bfloat16)
        up = (draw(experts, 2 * inter, width) / width ** 0.5).to(torch.bfloat16)
        down = (draw(experts, width, inter) / inter ** 0.5).to(torch.bfloat16)
        outs = []
        for tile_rows in (0, 256):
            outs.append(torch.full((n, width), float("nan"), device="cuda"))
            assert ops.experts_sorted(x, up, down, chosen, weights, outs[-1], tile_rows=tile_rows)
        assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])
