"""The 32-bit product for a few rows at the edges of its tiles, against the 64-bit product.

A result is a sum of K products in float32; split into 32 chains (eight wavefronts, four each) its error stays below
K / 32 + 8 roundings of 2^-24 in the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


@pytest.mark.parametrize("rows,outputs,inner,bias", [(1, 1, 512, False), (2, 3, 532, True), (8, 17, 644, False), (5, 1023, 580, True), (3, 1024, 2048, False),
                                                     (8, 4095, 636, True), (7, 4097, 516, False), (16, 16384, 512, True), (9, 16391, 772, False),
                                                     (2, 24, 9216, False)])
def test_few_rows_in_float32(ops, rows, outputs, inner, bias):
    print(f"few rows in float32 {rows} {outputs} {inner} {bias}", flush=True)
    generator = torch.Generator("cuda").manual_seed(rows + outputs)
    x, w, b = (torch.randn(*shape, device="cuda", generator=generator) for shape in ((rows, inner), (outputs, inner), (outputs,)))
    y = torch.full((rows, outputs), float("nan"), device="cuda")
    assert ops._linear_few_rows_float32(x, w, y, b if bias else None) is y
    exact = x.double() @ w.double().T + (b.double() if bias else 0.0)
    assert float((y - exact).norm() / exact.norm()) < (inner / 32 + 8) * 2.0 ** -24
    if ops._few_rows_float32(x, w, None):
        assert torch.equal(y, ops.linear(x, w, bias=b if bias else None))


def test_what_goes_to_the_library_as_before(ops):
    make = lambda *shape: torch.randn(*shape, device="cuda")
    for x, w in ((make(9, 512), make(100, 512)), (make(17, 512), make(20000, 512)), (make(2, 514), make(8, 514)), (make(512, 2).t(), make(8, 512)),
                 (make(2, 1024)[:, :512], make(8, 512)), (make(2, 512), make(512, 8).t()), (make(1026)[1:1025].view(2, 512), make(8, 512)),
                 (make(0, 512), make(8, 512)), (make(2, 508), make(8, 508))):
        assert not ops._few_rows_float32(x, w, None)
        exact = x.double() @ w.double().T
        assert float((ops.linear(x, w) - exact).norm()) <= 1e-5 * float(exact.norm())


def test_operands_that_do_not_fit_together_are_refused(ops):
    """What the kernel would read by address alone: a matrix or a result in host memory, matrices in a stack.  The library refuses them."""
    x, w = torch.randn(2, 512, device="cuda"), torch.randn(8, 512, device="cuda")
    assert ops._few_rows_float32(x, w, None)
    for weight, out in ((w.cpu(), None), (w, torch.empty(2, 8)), (torch.randn(8, 512, 3, device="cuda"), None)):
        assert not ops._few_rows_float32(x, weight, out)
        with pytest.raises((RuntimeError, ValueError)):
            ops.linear(x, weight, out=out)


def test_gradients_pass_through_the_32_bit_product(ops):
    x, w = torch.randn(2, 512, device="cuda", requires_grad=True), torch.randn(8, 512, device="cuda", requires_grad=True)
    ops.linear(x, w).sum().backward()
    exact = w.detach().double().sum(dim=0).expand(2, -1)
    assert float((x.grad - exact).norm()) <= 1e-6 * float(exact.norm())
    with torch.no_grad():
        assert ops._few_rows_float32(x, w, None)
