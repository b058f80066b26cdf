"""Rows of very different lengths that are shared out over one round although that rounds by many tiles, more splits asked for than a launch has use for, and
rows so long that one round's splits would not fit the paged kernel's tile table."""
import pytest

import test_gpu_ragged_rows as ragged
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu

CASES = [
    ([2000 + 1900 * i for i in range(16)], 16, 1, 4, ragged.SHARED),              # 32 splits for 16 rows: rounding costs 130 tiles
    ([16000] * 2 + [900 * (i + 1) for i in range(22)], 8, 1, 40, ragged.SHARED),   # asked for 7680 blocks
    ([10000 + 300 * (i % 5) for i in range(16)], 16, 1, 4, ragged.NSPLIT),       # rows much alike: several rounds
]


@pytest.mark.parametrize("lens,n_kv,G,nsplit,expect", CASES)
@pytest.mark.parametrize("path", [ragged.test_slot_cache, ragged.test_paged_pool])
def test_rows(path, lens, n_kv, G, nsplit, expect):
    require_gpu()
    path(lens, n_kv, G, nsplit, expect)


# 256 heads: sixteen splits a round for eight rows; 512: eight
@pytest.mark.parametrize("lens,n_kv", [
    ([60000] * 5 + [200] * 3, 32),        # a mean of more tiles than the table holds
    ([59200] * 3 + [16] * 5, 32),         # a mean of 694, but one round comes to 1234
    ([59200] * 2 + [16] * 6, 64),         # two rounds have two splits a row
])
def test_splits_stay_within_the_tile_table(lens, n_kv):
    """Rows whose one round would need splits of more than 1024 tiles: the paged launch makes four of each long row."""
    dev = require_gpu()
    import torch
    from test_gpu_long_row import splits_of
    gen, ns = torch.Generator(device=dev).manual_seed(3), 8
    layer, pool, bt, sl = ragged._paged(lens, n_kv, gen, dev)
    q = torch.randn(len(lens), n_kv, 128, generator=gen, device=dev).to(torch.bfloat16)
    q[0] = 0
    want = torch.cat([layer.attention(q[i:i + 1], pool, bt[i:i + 1], sl[i:i + 1], 4) for i in range(len(lens))]).float()
    for _ in range(2):
        ragged.assert_rows_close(layer.attention(q, pool, bt, sl, ns).float(), want)
        assert splits_of(layer._ws[(len(lens), n_kv, ns)], n_kv) == 4
    layer.check()
