"""Which router products leave the library (host code: no GPU needed)."""
import torch

from llmserver_amd.kernels import library
from llmserver_amd.kernels.ops import HipOps


def test_router_products_where_they_were_measured_to_be_faster():
    ops = HipOps.__new__(HipOps)
    ops._parts_libraries = {"experts": library.load("experts")}

    def parts(rows, experts, width, dtype):
        return ops._route_parts(torch.empty(rows, width, dtype=dtype), torch.empty(experts, width))
    for rows, experts, width in ((17, 64, 2048), (32, 256, 4096), (128, 128, 4096), (256, 64, 4096), (1024, 16, 2048)):
        assert parts(rows, experts, width, torch.bfloat16) == parts(rows, experts, width, torch.float32) == min(8, -(-width // 512))
    for rows, experts, width in ((256, 128, 2048), (512, 64, 2048), (4096, 8, 512)):
        assert parts(rows, experts, width, torch.bfloat16) and not parts(rows, experts, width, torch.float32)
    for dtype in (torch.bfloat16, torch.float32):
        assert not parts(1024, 64, 2048, dtype) and not parts(17, 64, 2044, dtype)
