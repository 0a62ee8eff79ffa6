"""The norm and gate of heads in its two forms, eight neighbouring numbers a lane and one, on both sides of every line between them (sizes, addresses, heads of up to 64 numbers
in few and in many pairs), with and without the read-out's denominators, against 64 bits.

Sums of `value_dim` squares in float32: 1e-5; bfloat16 results are rounded once more (2^-9)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens, heads, value_dim, offset", [(3, 16, 64, 0), (256, 16, 64, 0), (255, 16, 64, 0), (1, 1, 8, 0), (5, 3, 256, 0), (5, 3, 256, 1), (4, 5, 264, 0), (4, 5, 320, 0),
                                                              (7, 3, 100, 0), (6, 2, 33, 0), (40, 4, 128, 1)])
@pytest.mark.parametrize("below", [False, True])
def test_both_forms(dtype, tokens, heads, value_dim, offset, below):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    print(f"heads' norm {dtype} {tokens} {heads} {value_dim} {offset} {below}", flush=True)
    torch.manual_seed(tokens + value_dim)
    x, weight = torch.randn(tokens, heads * value_dim, device="cuda"), torch.randn(heads * value_dim, device="cuda")
    gate = torch.randn(tokens, heads * value_dim + 8, device="cuda").to(dtype)[:, offset:offset + heads * value_dim]      # (a view that begins at an odd place)
    under = torch.rand(tokens, heads, 2, device="cuda") - 0.3 if below else None
    out = torch.full((tokens, heads * value_dim), float("nan"), device="cuda", dtype=dtype)
    ops.heads_norm_gate(x, weight, True, 1e-6, gate, out, heads, value_dim, below=under, floor=1e-3 if below else 0.0)
    wide = x.double().view(tokens, heads, value_dim)
    if below:
        wide = wide / (torch.maximum(under[..., 0].abs(), under[..., 1]).double()[..., None] + 1e-3)
    g = gate.double().reshape(tokens, heads, value_dim)
    want = wide * torch.rsqrt(wide.pow(2).mean(dim=-1, keepdim=True) + 1e-6) * weight.double().view(heads, value_dim) * g * torch.sigmoid(g)
    close = dict(rtol=2.0 ** -8, atol=2.0 ** -9) if dtype == torch.bfloat16 else dict(rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(out.double().view_as(want), want, **close)
