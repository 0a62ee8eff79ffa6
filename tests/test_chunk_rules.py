"""Which steps run their recurrences and delta rules in chunks, and what becomes of those that cannot (host code: no GPU needed)."""
import types

import pytest
import torch

from llmserver_amd.kernels import library
from llmserver_amd.kernels.ops import HipOps
from llmserver_amd.parts.base import scratch_memory
from llmserver_amd.parts.recurrent import _chunk_scratch


@pytest.fixture()
def ops():
    made = HipOps.__new__(HipOps)
    made._parts_libraries = {name: library.load(name) for name in ("recurrent", "delta")}
    return made


def linear_bytes(ops, lengths, heads, dim, vdim):
    chunks = ops.linear_recurrence_chunks(sum(lengths), len(lengths), max(lengths), heads, dim, vdim)
    return 4 * heads * dim * (chunks * (vdim + 1) + sum(lengths)) if chunks else 0


def delta_bytes(ops, lengths, heads, dim, vdim):
    shape = ops.delta_rule_scratch(sum(lengths), len(lengths), max(lengths), heads, dim, vdim)
    return 4 * shape[0] * shape[1] * shape[2] if shape else 0


@pytest.mark.parametrize("bytes_of", [linear_bytes, delta_bytes])
def test_scratch_memory_has_a_bound_beyond_which_a_step_walks(ops, bytes_of):
    assert 0 < bytes_of(ops, [8192], 16, 128, 128) < 400e6
    for length in (8192, 16384, 32768, 65536, 262144):
        for heads, dim, vdim in ((16, 128, 128), (32, 128, 256), (64, 64, 64)):
            assert bytes_of(ops, [length], heads, dim, vdim) <= 1 << 30
    assert not bytes_of(ops, [262144], 16, 128, 128)


def test_a_step_without_room_for_scratch_memory_walks():
    def full(shape, dtype):
        raise torch.OutOfMemoryError("no room")
    asked = []
    rules = types.SimpleNamespace(linear_recurrence_chunks=lambda *shape: asked.append(shape) or 7)
    step = lambda empty: types.SimpleNamespace(ops=rules, row_len=torch.tensor([300, 1]), longest_row=lambda: 300, empty=empty)
    assert _chunk_scratch(step(full), 301, 2, 8, 16) == {}
    assert scratch_memory(step(full), {"scratch": (2, 3)}) == {}
    given = _chunk_scratch(step(lambda shape, dtype: torch.empty(shape, dtype=dtype)), 301, 2, 8, 16)
    assert {name: tuple(tensor.shape) for name, tensor in given.items()} == {"sums": (7, 2, 8, 16), "totals": (7, 2, 8), "queries": (301, 2, 8)}
    assert asked == [(301, 2, 300, 2, 8, 16)] * 2
