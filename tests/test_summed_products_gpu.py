"""Products of 17 to 64 rows in partial sums that a kernel adds up, with and without the gate's activation, against 64 bits, and what stays with the
library.  A sum of K products in float32 in a few dozen chains, rounded once to bfloat16: 2^-9 of each number, and 1e-5 of the result's size."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


def near(got, want):
    torch.testing.assert_close(got.double(), want, rtol=2.0 ** -8, atol=2e-5 * float(want.abs().max()))


@pytest.mark.parametrize("rows", [17, 31, 32, 33, 48, 64])
@pytest.mark.parametrize("outputs, inner", [(2816, 2048), (4096, 1024), (1028, 4088), (4100, 1400), (2048, 4096)])
def test_sums_of_partial_products(ops, rows, outputs, inner):
    print(f"summed products {rows} {outputs} {inner}", flush=True)
    torch.manual_seed(rows + outputs)
    x, w = torch.randn(rows, inner, device="cuda").bfloat16(), (torch.randn(outputs, inner, device="cuda") * inner ** -0.5).bfloat16()
    with torch.inference_mode():
        out = torch.full((rows, outputs), float("nan"), device="cuda", dtype=torch.bfloat16)
        assert (ops._partial_sums_to_add(x, w) is not None) == (rows <= 32 and 1 << 22 <= outputs * inner <= 1 << 23)
        assert ops.linear(x, w, out=out) is out
        near(out, x.double() @ w.double().T)
        if outputs % 8 == 0:
            assert ops._partial_sums_to_add(x, w, gated=True) is not None
            gate, up = (x.double() @ w.double().T).chunk(2, dim=1)
            near(ops.linear_gated(x, w), gate * torch.sigmoid(gate) * up)


@pytest.mark.parametrize("parts", [1, 2, 7, 8, 9, 17])
@pytest.mark.parametrize("rows, width", [(1, 8), (3, 1032), (17, 2056)])
def test_adding_up(ops, parts, rows, width):
    torch.manual_seed(parts + width)
    sums = torch.randn(parts, rows, width, device="cuda")
    out, gated = torch.full((rows, width), float("nan"), device="cuda", dtype=torch.bfloat16), torch.full((rows, width // 2), float("nan"), device="cuda", dtype=torch.bfloat16)
    lib, stream = ops._elementwise, torch.cuda.current_stream().cuda_stream
    total = sums.double().sum(dim=0)
    assert lib.lsa_sum_parts(sums.data_ptr(), parts, out.data_ptr(), rows, width, stream) == 0
    near(out, total)
    gate, up = total.chunk(2, dim=1)
    for activation, act in ((0, gate * torch.sigmoid(gate)), (1, 0.5 * gate * (1 + torch.tanh(0.7978845608028654 * (gate + 0.044715 * gate ** 3))))):
        assert lib.lsa_gated_parts(sums.data_ptr(), parts, gated.data_ptr(), rows, width // 2, activation, stream) == 0
        near(gated, act * up)
    assert lib.lsa_sum_parts(sums.data_ptr(), parts, out.data_ptr(), rows, 6, stream) != 0 and lib.lsa_sum_parts(sums.data_ptr() + 4, parts, out.data_ptr(), rows, width, stream) != 0


def test_what_stays_with_the_library(ops):
    make = lambda *shape: torch.randn(*shape, device="cuda").bfloat16()
    with torch.inference_mode():
        for x, w in ((make(16, 2048), make(2816, 2048)), (make(33, 2048), make(2816, 2048)), (make(20, 2048), make(1024, 2048)), (make(20, 2048), make(6144, 2048)),
                     (make(20, 4096)[:, :2048], make(2816, 2048)), (make(20, 2048).float(), make(2816, 2048).float()), (make(2048, 20).t(), make(2816, 2048)),
                     (make(20 * 2048 + 1)[1:].view(20, 2048), make(2816, 2048))):
            assert ops._partial_sums_to_add(x, w) is None
    x, w = make(20, 2048).requires_grad_(), make(2816, 2048)
    assert ops._partial_sums_to_add(x, w) is None
    ops.linear(x, w).float().sum().backward()
    assert x.grad is not None
