"""Which steps run their recurrences and delta rules in chunks, and what becomes of those that cannot (host code: no GPU needed)."""
import types

import pytest
import torch

from llmserver_amd.engine.batch import StepEntry
from llmserver_amd.engine.replay import make_runner
from llmserver_amd.kernels import library
from llmserver_amd.kernels.ops import HipOps
from llmserver_amd.parts.base import scratch_memory
from llmserver_amd.parts.recurrent import _chunk_scratch
from torch_ops import TorchOps


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


# (rows' lengths, heads, key channels, value channels): where the chunks were measured to be faster than the walk, and where they were not
CHUNKS_OF_LINEAR = [([144], 16, 128, 128), ([160] * 4, 16, 128, 128), ([2048], 8, 128, 256), ([2048] * 8, 16, 128, 128), ([256] * 2, 16, 128, 128), ([512] * 4, 16, 128, 128), ([512] + [1] * 16, 16, 128, 128),
                    ([128] * 4, 16, 64, 64), ([512] * 8, 16, 64, 64), ([512] * 4, 32, 64, 64), ([512] * 8, 8, 96, 192), ([256] * 16, 8, 96, 192)]
WALKS_OF_LINEAR = [([100], 16, 128, 128), ([112], 16, 128, 128), ([256] * 4, 16, 128, 128), ([96], 16, 64, 64), ([8] * 4 + [0], 16, 64, 64),
                   ([100], 32, 128, 128), ([64], 16, 64, 64), ([64] * 16, 16, 128, 128), ([32] * 32, 16, 64, 64), ([128] * 8, 16, 128, 128),
                   ([256] * 16, 16, 64, 64), ([1] * 40, 16, 128, 128), ([112] + [1] * 64, 16, 128, 128), ([128] + [1] * 8, 16, 128, 128), ([512] * 16, 16, 128, 128),
                   ([1024] * 8, 16, 128, 128), ([2048] * 16, 16, 64, 64)]
CHUNKS_OF_DELTA = [([512], 16, 128, 128), ([1900], 16, 128, 128), ([512] * 4, 16, 128, 128), ([512] + [1] * 16, 16, 128, 128), ([256], 16, 64, 64),
                   ([2048], 32, 64, 64), ([1024] + [64] * 8, 32, 128, 128), ([512] * 4, 8, 96, 192)]
WALKS_OF_DELTA = [([192], 4, 128, 128), ([160], 16, 128, 128), ([256], 32, 128, 128), ([256] * 8, 4, 128, 128), ([256] * 4, 16, 128, 128), ([64] * 16, 16, 128, 128),
                  ([512] * 16, 16, 128, 128), ([512] * 16, 8, 128, 256), ([512] * 16, 16, 64, 64), ([256] + [1] * 16, 16, 128, 128), ([1] * 40, 16, 128, 128)]


def test_steps_run_the_way_that_was_measured_to_be_faster(ops):
    for case in CHUNKS_OF_LINEAR:
        assert linear_bytes(ops, *case), case
    for case in WALKS_OF_LINEAR:
        assert not linear_bytes(ops, *case), case
    for case in CHUNKS_OF_DELTA:
        assert delta_bytes(ops, *case), case
    for case in WALKS_OF_DELTA:
        assert not delta_bytes(ops, *case), case


# rows' lengths of steps that would be filled up to the same number of tokens and rows: (in chunks, token by token) by the rule of 16 heads of 128 x 128
@pytest.mark.parametrize("design,rule,in_chunks,walked", [
    ("barotar", "linear_recurrence_chunks", [[490] + [1] * 15, [300] + [12] * 15], [[32] * 16, [60] + [30] * 15]),
    ("gogalix", "delta_rule_scratch", [[490] + [1] * 15], [[32] * 16]), ("gogalix", "delta_rule_scratch", [[478, 1, 1]], [[160] * 3])])
def test_captured_steps_choose_by_their_longest_row(ops, design, rule, in_chunks, walked):
    """A graph is shared by steps that choose alike only, and each step chooses as it would if it were not captured."""
    import tiny_barotar, tiny_gogalix
    tiny = {"barotar": tiny_barotar, "gogalix": tiny_gogalix}[design]
    twins = TorchOps()
    setattr(twins, rule, lambda n_tokens, rows, longest, *sizes: getattr(ops, rule)(n_tokens, rows, longest, 16, 128, 128))
    name = next(iter(tiny.CASES))
    runner = make_runner(tiny.model_folder(name), "float32", 4096, tiny.CASES[name][2], device="cpu", ops=twins, max_live=16)
    runner.use_graphs, runner._host_bounds_a_step = True, lambda tokens, keys: True         # (only the keys are asked for)
    for row in range(16):
        runner.cache.open(row)
    keys = {}
    for lengths in in_chunks + walked:
        entries = [StepEntry(row, [1] * length, [length - 1]) for row, length in enumerate(lengths)]
        runner._graph_key(entries)
        keys[tuple(lengths)] = key = runner._graph_key(entries)
        step = runner.build_context(entries, filler_rows=key[1] - 1 - len(entries), filler_tokens=key[2] - sum(lengths) - (key[1] - 1 - len(entries)))
        step.static_max_keys = 4096
        assert step.n_tokens == key[2] and step.longest_row() == max(int(length) for length in step.h_row_len)
        eager = bool(getattr(ops, rule)(step.n_tokens, step.n_rows, step.longest_row(), 16, 128, 128))
        assert eager == (lengths in in_chunks) == key[5][-1], lengths
    assert len({key[:3] for key in keys.values()}) == 1 and len(set(keys.values())) == 2
