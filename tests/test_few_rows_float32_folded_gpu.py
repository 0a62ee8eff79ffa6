"""The 32-bit products of up to 8 rows whose steps take 32 inner indices, at the edges of steps, of trips and of a workgroup's rows of the weight, against 64 bits.

A result is a sum of K products in 32 chains (eight wavefronts, four each), twice as many where a step's halves have their own, which is up to 8 rows with up to 8 rows of the weight a
workgroup: its error stays below K / chains + 9 roundings of 2^-24 in the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llmserver_amd.kernels import default_ops
    return default_ops()


def drawn(rows, outputs, inner):
    generator = torch.Generator("cuda").manual_seed(rows + outputs + inner)
    return torch.randn(rows, inner, device="cuda", generator=generator), torch.randn(outputs, inner, device="cuda", generator=generator) * inner ** -0.5


def chains(rows, outputs):
    """As many as ``few_f32_rows`` in ``csrc/gemm.hip`` leaves: sixteen rows of the weight a workgroup, or more than 8 of the other operand, have no halves."""
    sixteen = outputs >= 8192 or outputs >= 4096 and rows > (8 if outputs >= 6144 else 4)
    return 32 if rows > 8 or sixteen else 64


def error(got, exact):
    return float((got.double() - exact).norm() / exact.norm())


# one trip of 4, 6 and 8 steps to their last number and one behind it, two of 6 and of 8; rows of the weight around 4, 8 and 16 a workgroup
@pytest.mark.parametrize("inner", [4, 28, 512, 1020, 1024, 1028, 1536, 1540, 2048, 2052, 3072, 3076, 4100])
@pytest.mark.parametrize("rows, outputs", [(1, 1), (8, 5), (2, 1024), (7, 1025), (4, 4095), (4, 4097), (5, 4096), (8, 6145), (3, 8191), (9, 1023), (16, 1030)])
def test_steps_of_32(ops, rows, outputs, inner):
    print(f"float32 folded {rows} {outputs} {inner}", flush=True)
    x, w = drawn(rows, outputs, inner)
    x[:, -1] = 1e3                                                # (the last inner index counts once)
    y = torch.full((rows, outputs), float("nan"), device="cuda")
    assert ops._linear_few_rows_float32(x, w, y) is y
    assert error(y, x.double() @ w.double().T) < (inner / chains(rows, outputs) + 9) * 2.0 ** -24


@pytest.mark.parametrize("rows, pairs, inner", [(1, 3, 512), (8, 511, 1028), (2, 512, 768), (4, 2047, 1024), (4, 2049, 800), (5, 2050, 900), (8, 3073, 1024), (6, 4096, 1024)])
def test_gate_and_up_rows_beside_each_other(ops, rows, pairs, inner):
    print(f"float32 folded gated {rows} {pairs} {inner}", flush=True)
    x, w = drawn(rows, 2 * pairs, inner)
    got = torch.full((rows, pairs), float("nan"), device="cuda")
    assert ops._gemm.lsa_gemm_few_f32_gated(x.data_ptr(), w.data_ptr(), got.data_ptr(), rows, pairs, inner, None, 0, 0.0, torch.cuda.current_stream().cuda_stream) == 0
    gate, up = (x.double() @ w.double().T).chunk(2, dim=1)
    assert error(got, gate * torch.sigmoid(gate) * up) < 2 * (inner / chains(rows, 2 * pairs) + 9) * 2.0 ** -24          # (two products meet)


@pytest.mark.parametrize("rows, outputs, inner", [(1, 1024, 3072), (4, 2048, 6144), (2, 1020, 2048), (8, 1028, 1024)])
def test_the_stream_update_of_folded_products(ops, rows, outputs, inner):
    print(f"float32 folded stream {rows} {outputs} {inner}", flush=True)
    x, w = drawn(rows, outputs, inner)
    resid, norm_weight = drawn(rows, 2, outputs)[0], torch.rand(outputs, device="cuda") + 0.5
    stream, weighted, squares = ops.linear_into_stream(x, w, resid, norm_weight)
    assert error(stream, resid.double() + x.double() @ w.double().T) < (inner / chains(rows, outputs) + 9) * 2.0 ** -24
    assert torch.equal(weighted, stream * norm_weight) and squares.shape[1] <= ops.SCALE_PARTS
    assert error(squares.sum(dim=1), (stream.double() ** 2).sum(dim=1)) < 16 * 2.0 ** -24
