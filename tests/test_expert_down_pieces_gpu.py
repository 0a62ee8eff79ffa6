"""The second product of experts pair by pair where a token's rows end inside the pieces that a lane asks for ahead, with identity experts among the choices."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (choices, numbers of a hidden row): one to nine trips of 64 pieces of 16 bytes, whole and not, in ones, threes and fours; rows of one piece (of 4 or 8 numbers)
@pytest.mark.parametrize("top,inter", [(1, 8), (2, 8), (7, 8), (3, 4), (1, 504), (2, 256), (3, 344), (2, 768), (4, 512), (5, 408), (3, 1408), (8, 72), (6, 704), (2, 2304), (9, 512)])
@pytest.mark.parametrize("tokens", [1, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_that_end_between_pieces(dtype, tokens, top, inter):
    """32-bit sums of `terms` products are off by at most (terms + 64) 2^-24 of the sum of their sizes (the weights' product, the lanes' sums).  Expert 0 holds no numbers
    and is nobody's choice: a piece behind the last one, or an identity expert's, must not count."""
    from llmserver_amd.kernels import default_ops
    print(f"expert down {dtype} {tokens} {top} {inter}", flush=True)
    ops, width, experts = default_ops(), 40, 10
    generator = torch.Generator("cuda").manual_seed(inter + top)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=generator)
    down = draw(experts, width, inter).to(dtype)
    down[0] = float("nan")
    chosen = torch.stack([1 + torch.randperm(experts - 1, generator=torch.Generator().manual_seed(t))[:top] for t in range(tokens)]).to(torch.int32).cuda()
    chosen[-1, -1] = experts + 1                                   # an identity expert
    hidden, weights, x, out = draw(tokens * top, inter).to(dtype), draw(tokens, top), draw(tokens, width).to(dtype), torch.full((tokens, width), float("nan"), device="cuda")
    ops.experts_down(hidden, down, chosen, weights, out, x=x)
    want, sizes = torch.zeros(tokens, width, device="cuda", dtype=torch.float64), torch.zeros(tokens, width, device="cuda", dtype=torch.float64)
    for t in range(tokens):
        for s in range(top):
            e = int(chosen[t, s])
            w, h = weights[t, s].double(), hidden[t * top + s].double()
            want[t] += w * (x[t].double() if e >= experts else down[e].double() @ h)
            sizes[t] += w.abs() * (x[t].double().abs() if e >= experts else down[e].double().abs() @ h.abs())
    assert bool(((out.double() - want).abs() <= (top * inter + 64) * 2.0 ** -24 * sizes).all())
