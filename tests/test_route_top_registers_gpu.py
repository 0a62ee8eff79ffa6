"""Choices of experts out of registers (up to 128 experts in one group): the very numbers of the kernel for any number of experts, which is made to
take the same logits by experts beyond 128 that nobody can choose."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts, top", [(1, 1), (2, 2), (63, 6), (64, 6), (65, 8), (72, 6), (127, 64), (128, 1)])
@pytest.mark.parametrize("scoring", [0, 1, 2])
@pytest.mark.parametrize("parts", [1, 3, 8])
def test_same_choices_and_weights(experts, top, scoring, parts):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    lib = ops._part_library("experts")
    print(f"route top {experts} {top} {scoring} {parts}", flush=True)
    g = torch.Generator("cuda").manual_seed(experts * 7 + top + scoring)
    tokens, gate = 9, scoring == 2
    logits = torch.randn(parts, tokens, experts + 1, device="cuda", generator=g)
    logits[:, 1] = logits[:, 1, :1]                       # equal logits: the lowest index first
    logits[:, 2, :experts // 2] = -torch.inf
    logits[:, 3] = -torch.inf
    logits[0, 4, experts // 3] = torch.nan
    extra = torch.randn(experts, device="cuda", generator=g) * 0.01
    bias, correction = (extra, None) if scoring < 2 else (None, extra)
    ptr = lambda tensor: None if tensor is None else tensor.data_ptr()
    def run(logits, count, bias, correction):
        chosen = torch.full((tokens, top), -7, device="cuda", dtype=torch.int32)
        weights, gates = torch.full((tokens, top), torch.nan, device="cuda"), torch.full((tokens,), torch.nan, device="cuda")
        stream = torch.cuda.current_stream().cuda_stream
        assert lib.lsa_route_top(ptr(logits), count, top, ptr(chosen), ptr(weights), tokens, scoring, 1, 1, ptr(bias), ptr(correction), 1.5, count + 1,
                                 ptr(gates) if gate else None, parts, stream) == 0
        return chosen, weights, gates
    got = run(logits.contiguous(), experts, bias, correction)
    more = 200 - experts                                  # the same experts and some that come last: that kernel's way
    padded = torch.cat([logits[..., :experts], torch.full((parts, tokens, more), -torch.inf, device="cuda"), logits[..., experts:]], dim=-1).contiguous()
    longer = lambda tensor: None if tensor is None else torch.cat([tensor, torch.full((more,), -10.0, device="cuda")])
    want = run(padded, 200, longer(bias), longer(correction))
    ordinary = [row for row in range(tokens) if row not in (2, 3, 4)] if top > experts // 2 else [row for row in range(tokens) if row not in (3, 4)]
    assert torch.equal(got[0][ordinary], want[0][ordinary])
    if gate:
        assert torch.equal(got[2], want[2])
    torch.testing.assert_close(got[1][ordinary], want[1][ordinary], atol=0, rtol=1e-6 if scoring == 2 else 0)     # (the softmax's sum is in another order)
    assert ((got[0] >= 0) & (got[0] < experts)).all()
