"""Which steps of one token a row behind short contexts go to the kernel of their own: those whose workgroups each have a compute unit (two to a
unit in float32), and beyond that the forms that were measured to stay faster (host code: no GPU needed)."""
import pytest
import torch

from llmserver_amd.kernels.ops import HipOps
from llmserver_amd.parts.attention import AttentionTuning

BF16, F32 = torch.bfloat16, torch.float32


@pytest.fixture(scope="module")
def ops():
    made = HipOps.__new__(HipOps)
    made.attention_tuning_for = lambda dtype, head_dim=None: AttentionTuning(target_waves=4 * 256)
    return made


@pytest.mark.parametrize("dtype, n_q, n_kv, head_dim, most_rows", [(BF16, 16, 8, 128, 32), (BF16, 32, 8, 128, 32), (BF16, 64, 4, 128, 64), (BF16, 16, 8, 32, 32),
                                                                   (BF16, 40, 2, 128, 64), (F32, 16, 8, 128, 64), (F32, 8, 8, 128, 64), (BF16, 12, 1, 128, 256)])
def test_workgroups_with_a_compute_unit_each(ops, dtype, n_q, n_kv, head_dim, most_rows):
    assert all(ops.single_tokens_pay(dtype, head_dim, rows, n_q, n_kv) for rows in (1, most_rows // 2 + 1, most_rows))
    assert not any(ops.single_tokens_pay(dtype, head_dim, rows, n_q, n_kv) for rows in (most_rows + 1, 4 * most_rows))


def test_forms_that_stay_faster_beyond_that(ops):
    for dtype, n_q, n_kv, head_dim in ((BF16, 64, 4, 256), (BF16, 24, 2, 192), (BF16, 40, 2, 96), (F32, 16, 4, 256), (F32, 8, 8, 64), (F32, 16, 16, 32)):
        assert ops.single_tokens_pay(dtype, head_dim, 2048, n_q, n_kv)
    assert not ops.single_tokens_pay(F32, 64, 65, 8, 8, plain=False) and ops.single_tokens_pay(F32, 64, 64, 8, 8, plain=False)
    assert not ops.single_tokens_pay(F32, 64, 65, 16, 8)
