"""The router's own product for steps of more than a few tokens, in partial sums that the choice adds up."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,experts,top,width", [(17, 5, 5, 8), (33, 17, 3, 520), (64, 130, 8, 2048), (40, 16, 2, 4104), (20, 65, 64, 1000),
                                                    (18, 100, 70, 136), (300, 64, 6, 2048), (600, 64, 6, 2048)])
@pytest.mark.parametrize("scoring", ["softmax", "sigmoid", "softmax_all"])
def test_choices_from_partial_sums(ops, dtype, rows, experts, top, width, scoring):
    """Edges of the tiles of 16 x 16 and of the ranges of the width, one range and eight, more choices than lanes, and a step too large for
    the kernel.  A dot product of `width` numbers in 32 bits is off by at most width * 2^-24 times the sum of its terms' sizes (the
    kernel's partial sums are shorter than that): a choice may differ from the exact one by twice that."""
    print(f"route parts {dtype} {rows} {experts} {top} {width} {scoring}", flush=True)
    generator = torch.Generator("cuda").manual_seed(rows)
    x = torch.randn(rows, width, device="cuda", generator=generator).to(dtype)
    router = torch.randn(experts + 1, width, device="cuda", generator=generator) * width ** -0.5
    chosen = torch.empty(rows, top, dtype=torch.int32, device="cuda")
    weights, gate = torch.empty(rows, top, device="cuda"), torch.empty(rows, device="cuda")
    taken = ops._route_parts(x, router)
    assert bool(taken) == (rows < (600 if dtype == torch.bfloat16 else 300))
    ops.route_experts(x, router, top, chosen, weights, scoring=scoring, gate_out=gate)
    exact = x.double() @ router.double().T
    bound = float((x.double().abs() @ router.double().abs().T).max()) * width * 2.0 ** -24
    logits, picked = exact[:, :experts], exact[:, :experts].gather(1, chosen.long())
    assert int(torch.stack([row.unique().numel() == torch.tensor(top) for row in chosen]).sum()) == rows
    assert bool(((picked - logits.topk(top, dim=1).values).abs() <= 2 * bound).all())
    if scoring == "softmax":
        want = torch.softmax(picked, dim=1)
    elif scoring == "sigmoid":
        want = torch.sigmoid(picked)
    else:
        scores = torch.softmax(logits, dim=1).gather(1, chosen.long())
        want = scores / scores.sum(dim=1, keepdim=True)
    # (a change of d in every logit changes such a weight by a factor of at most e^(2 d); the functions themselves a few units in the last place)
    assert bool(((weights.double() - want).abs() <= (4 * bound + 1e-5) * want).all())
    assert bool(((gate.double() - torch.sigmoid(exact[:, experts])).abs() <= bound + 1e-6).all())
