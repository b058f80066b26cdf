"""Ragged rows in one round of four-wave blocks, ordered by the size of their splits with the later half of the launch running backwards: rows across the
middle, odd counts of splits, equal sizes, empty rows, as many rows as a wave has lanes; and just outside the rule."""
import pytest

import test_gpu_ragged_rows as ragged
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu

CASES = [
    ([9000] + [2000 + 100 * (i // 4) for i in range(31)], 8, 2, 2),        # equal sizes, one row of several splits
    ([0, 1, 16, 17] + [700 * i + 5 for i in range(1, 27)], 5, 1, 4),       # 102 splits at most, empty and tiny rows
    ([12800 - 880 * i for i in range(14)], 16, 1, 3),                     # 32 splits, blocks left over at the launch's end
    ([12000] * 3 + [300] * 15, 16, 2, 2),                                  # rows of several splits, all alike, then whole rows
    ([50 + 160 * ((37 * i) % 64) for i in range(64)], 3, 4, 2),            # 128 splits of 64 rows
    ([50 + 160 * ((37 * i) % 65) for i in range(65)], 3, 4, 2),            # more rows than lanes
    ([400 * (1 + i % 7) for i in range(30)], 8, 1, 2),                     # splits about as short as the rule takes
]


@pytest.mark.parametrize("lens,n_kv,G,nsplit", CASES)
@pytest.mark.parametrize("path", [ragged.test_slot_cache, ragged.test_paged_pool])
def test_order(path, lens, n_kv, G, nsplit):
    require_gpu()
    path(lens, n_kv, G, nsplit, ragged.SHARED)
