import numpy as np
import pytest

from async_llm_amd.shared_cache.block_ops import slots_meet


@pytest.mark.parametrize("a, b, meet", [
    ([0], [0], True),
    ([0], [1], False),
    ([5, 9, 7], [8, 6, 9], True),
    ([5, 9, 7], [8, 6, 10], False),
    ([-3, 4], [-3], True),
    ([-3, 4], [3, -4], False),
    ([0, 1 << 40], [1 << 40], True),  # sorted: too wide to mark
    ([0, 1 << 40], [1, (1 << 40) - 1], False),
    ([-(1 << 63), 0], [(1 << 63) - 1], False),
])
def test_slots_meet(a, b, meet):
    assert slots_meet(np.array(a, dtype=np.int64), np.array(b, dtype=np.int64)) is meet
