"""Updates of several streams in steps of many rows: rows that are kept whole one column a load are taken so (the numbers of rows at any address), longer ones four at
a time, against 64 bits.  Sums of `width` squares in float32: 5e-6; bfloat16 results are rounded once more (2^-9)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("streams", [1, 2, 4])
@pytest.mark.parametrize("rows, width", [(512, 2048), (513, 2048), (513, 1028), (520, 2052), (513, 1024)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_updates_of_many_rows(streams, rows, width, dtype):
    from llmserver_amd.kernels import default_ops
    ops = default_ops()
    print(f"stream updates {streams} {rows} {width} {dtype}", flush=True)
    torch.manual_seed(rows + width)
    values = torch.randn(streams * rows * width + 1, device="cuda")
    y = torch.randn(rows, width, device="cuda").to(dtype)
    read, mix, write, weight = torch.randn(streams, device="cuda"), torch.randn(streams, streams, device="cuda"), torch.randn(streams, device="cuda"), torch.randn(width, device="cuda")
    def run(offset):
        x = torch.empty(streams * rows * width + offset, device="cuda")[offset:].view(streams, rows, width).copy_(values[1:].view(streams, rows, width))
        out = torch.full((rows, width), float("nan"), device="cuda", dtype=dtype)
        ops.streams_update(x, y, mix, write, read, weight, 1e-6, out)
        return x, out
    (x, out), (shifted, shifted_out) = run(0), run(1)
    fresh = torch.einsum("st,snw->tnw", mix.double(), values[1:].view(streams, rows, width).double()) + write.double()[:, None, None] * y.double()
    summed = torch.einsum("s,stw->tw", read.double(), fresh)
    normed = summed * torch.rsqrt(summed.pow(2).mean(dim=-1, keepdim=True) + 1e-6) * weight.double()
    torch.testing.assert_close(x.double(), fresh, rtol=5e-6, atol=5e-6)
    torch.testing.assert_close(out.double(), normed, **(dict(rtol=2.0 ** -8, atol=1e-3) if dtype == torch.bfloat16 else dict(rtol=5e-6, atol=5e-6)))
    assert torch.equal(x, shifted)
    if 512 < rows and 1024 < width <= 2048:
        assert torch.equal(out, shifted_out)               # the same way through the row: equal bits
