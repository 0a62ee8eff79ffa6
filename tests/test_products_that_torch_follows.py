"""Products that somebody follows (autograd, tangents of forward-mode differentiation, vmap, tracing, dispatch modes) stay calls of torch: a kernel that takes
addresses would fail there or lose what is followed.  The question itself on the CPU; the products on the GPU."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils.flop_counter import FlopCounterMode


def test_who_follows_a_call():
    from llmserver_amd.kernels.ops import _followed
    x, seen = torch.randn(3, 4), []
    ask = lambda a: (seen.append(_followed(a)), a * 2.0)[1]
    assert not _followed(x, None, torch.nn.Parameter(x, requires_grad=False))
    torch.vmap(ask)(x)
    torch.func.jvp(ask, (x,), (x,))
    torch.func.grad(lambda a: ask(a).sum())(x)
    make_fx(ask)(x)
    torch.jit.trace(ask, x, check_trace=False)
    with FlopCounterMode(display=False):
        ask(x)
    with forward_ad.dual_level():
        ask(forward_ad.make_dual(x, x))
        assert not _followed(x)
    ask(x.clone().requires_grad_())
    assert len(seen) == 8 and all(seen)
    with torch.no_grad():
        assert not _followed(x.clone().requires_grad_())


@pytest.mark.gpu
@pytest.mark.parametrize("rows, outputs, inner, dtype", [(20, 2816, 2048, torch.bfloat16), (4, 1024, 1024, torch.float32)])
def test_products_keep_their_tangents_and_transforms(rows, outputs, inner, dtype):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    print(f"followed products {rows} {outputs} {inner} {dtype}", flush=True)
    torch.manual_seed(rows)
    x, tangent = torch.randn(rows, inner, device="cuda").to(dtype), torch.randn(rows, inner, device="cuda").to(dtype)
    w = (torch.randn(outputs, inner, device="cuda") * inner ** -0.5).to(dtype)
    takes = lambda a: ops._partial_sums_to_add(a, w) is not None or ops._few_rows_float32(a, w, None)
    assert takes(x)
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(x, tangent)
        assert not takes(dual)
        y = forward_ad.unpack_dual(ops.linear(dual, w))
        assert torch.equal(y.primal, torch.mm(x, w.t())) and torch.equal(y.tangent, torch.mm(tangent, w.t()))
    asked = []
    torch.vmap(lambda a: (asked.append(takes(a)), a)[1])(torch.stack([x, tangent]))
    assert asked == [False]
    if dtype == torch.float32:
        both = torch.vmap(lambda a: ops.linear(a, w))(torch.stack([x, tangent]))
        torch.testing.assert_close(both[1], torch.mm(tangent, w.t()), rtol=1e-5, atol=1e-5)
        resid, norm = torch.randn(rows, outputs, device="cuda"), torch.ones(outputs, device="cuda")
        assert ops.linear_into_stream(x, w, resid, norm) is not None and ops.linear_into_stream(x, w, resid.requires_grad_(), norm) is None
    torch.cuda.synchronize()


def test_products_on_another_gpu_than_the_current_one(monkeypatch):
    from llmserver_amd.kernels.ops import _on_current_gpu

    class On:
        def __init__(self, index):
            self.device = torch.device("cuda", index)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    assert _on_current_gpu(On(0), None, On(0)) and not _on_current_gpu(On(1)) and not _on_current_gpu(On(0), On(1))
