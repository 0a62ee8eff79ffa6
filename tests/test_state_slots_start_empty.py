"""A state slot that a request gets holds zeros in every mixer's pool, whatever the pools' shapes and types, and other slots stay as they are."""
import pytest
import torch

from llmserver_amd.cache.manager import CacheManager
from llmserver_amd.parts.base import StateSpec


@pytest.mark.parametrize("specs", [[((3,), "float32")], [((2, 4), "float32"), ((5,), "bfloat16"), ((2, 4), "float32"), ((1, 1, 7), "float32")]])
def test_a_slot_starts_empty(specs):
    manager = CacheManager({i: StateSpec(shape, dtype) for i, (shape, dtype) in enumerate(specs)}, num_pages=0, page_size=16, dtype=torch.float32,
                           device=torch.device("cpu"), num_state_slots=3)
    for tensor in manager.state.values():
        tensor.fill_(7.0)
    slot = manager.open("a").state_slot
    for tensor in manager.state.values():
        assert not tensor[slot].any()
        assert all((tensor[other] == 7.0).all() for other in range(4) if other != slot)


def test_a_manager_that_only_plans_has_nothing_to_clear():
    manager = CacheManager({0: StateSpec((3,))}, 16, 0, num_state_slots=1, allocate_storage=False)
    assert manager.open("a").state_slot == 0
