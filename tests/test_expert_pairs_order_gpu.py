"""Experts pair by pair, whatever numbers of tokens, experts chosen and columns the workgroups' order on the chip has to cover (blocks of columns
that are no multiple of the eight XCDs, one token, shared and identity experts): every output is written, and is the 64-bit one.

Sums of `width` products in 32 bits, hidden rows rounded once to bfloat16 (2^-9): 1e-2 of the result; float32: (width + inter) roundings, 1e-5."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens, top, experts, inter, width, identity, shared", [(1, 1, 2, 8, 8, 0, 0), (1, 6, 64, 132, 260, 0, 0), (8, 6, 64, 1408, 512, 0, 0),
                                                                                  (3, 2, 5, 17, 40, 2, 0), (4, 3, 9, 100, 72, 0, 300), (7, 1, 3, 16, 36, 0, 0)])
def test_every_column_of_every_pair(dtype, tokens, top, experts, inter, width, identity, shared):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    print(f"expert pairs {dtype} {tokens} {top} {experts} {inter} {width} {identity} {shared}", flush=True)
    g = torch.Generator("cuda").manual_seed(tokens * 100 + width)
    make = lambda *shape: torch.randn(*shape, device="cuda", generator=g)
    x, gate_up, down = make(tokens, width).to(dtype), (make(experts, 2 * inter, width) * width ** -0.5).to(dtype), (make(experts, width, inter) * inter ** -0.5).to(dtype)
    chosen = torch.stack([torch.randperm(experts + identity, device="cuda", generator=g)[:top] for _ in range(tokens)]).to(torch.int32)
    weights = torch.softmax(make(tokens, top), dim=-1)
    hidden, out = torch.full((tokens * top, inter), float("nan"), device="cuda", dtype=dtype), torch.full((tokens, width), float("nan"), device="cuda")
    beside, after = {"identity": identity} if identity else {}, {"x": x} if identity else {}
    if shared:
        sgu, sd, sh = (make(2 * shared, width) * width ** -0.5).to(dtype), (make(width, shared) * shared ** -0.5).to(dtype), torch.full((tokens, shared), float("nan"), device="cuda", dtype=dtype)
        beside["shared"], after["shared"] = (sgu, sh), (sd, sh)
    ops.experts_gate_up(x, gate_up, chosen, hidden, **beside)
    ops.experts_down(hidden, down, chosen, weights, out, **after)
    def expert(row, gu, d, size):
        gate, up = gu.double() @ row, None
        gate, up = gate[:size], gate[size:]
        return d.double() @ (gate * torch.sigmoid(gate) * up)
    want = torch.stack([sum(float(weights[t, s]) * (x[t].double() if e >= experts else expert(x[t].double(), gate_up[e], down[e], inter))
                            for s, e in enumerate(chosen[t].tolist())) + (expert(x[t].double(), sgu, sd, shared) if shared else 0.0) for t in range(tokens)])
    assert float((out.double() - want).norm() / want.norm()) < (1e-5 if dtype == torch.float32 else 1e-2)
