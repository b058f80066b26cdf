"""One row much longer than the others in a batch that fills the chip by itself: the long row's splits, and the results."""
import pytest
import torch

import test_gpu_ragged_rows as ragged
from common import assert_rows_close
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu

# lengths, kv heads, splits asked for; splits of the longest row, at least
CASES = [
    ([2000] * 31 + [16000] + [2000] * 32, 8, 2, 6),            # one round has a unit for each row
    ([2000] * 31 + [16000] + [2000] * 32, 8, 4, 6),
    ([16000] + [2000] * 61, 8, 2, 6),                           # ... and two more
    ([1000] * 15 + [9000] + [1000] * 16, 16, 4, 6),
    ([600] * 100 + [9000] + [600] * 99, 2, 2, 8),               # more rows than a wave has lanes
    ([600] * 100 + [9000] + [600] * 99, 2, 3, 8),
    ([16 * i + 1 for i in range(60)] + [40000], 8, 3, 12),      # short ones of all lengths
]


def splits_of(ws, n_q):
    """How many splits a row of all-zero queries got: its largest scores are zeros."""
    zero = int(((ws.pm >> 32 == int(ws.epoch[0])) & (ws.pm & 0x7FFFFFFF == 0)).sum())
    assert zero % n_q == 0 and ws.failure_bits() == 0
    return zero // n_q


def _queries(lens, n_q, gen, dev):
    q = torch.randn(len(lens), n_q, 128, generator=gen, device=dev).to(torch.bfloat16)
    q[lens.index(max(lens))] = 0
    return q


@pytest.mark.parametrize("lens,n_kv,nsplit,least", CASES)
def test_slot_cache(lens, n_kv, nsplit, least):
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    gen = torch.Generator(device=dev).manual_seed(len(lens))
    cache = CompressedKVCache(len(lens), n_kv, max(lens) + 16, device=dev)
    for i, L in enumerate(lens): cache.prefill(i, ragged._rows(gen, L, n_kv, dev), ragged._rows(gen, L, n_kv, dev))
    q, slots = _queries(lens, n_kv, gen, dev), torch.arange(len(lens), dtype=torch.int32, device=dev)
    want = torch.cat([cache.attention(q[i:i + 1], slots[i:i + 1], ragged.SCALE, nsplit=7) for i in range(len(lens))]).float()
    for _ in range(2):
        assert_rows_close(cache.attention(q, slots, ragged.SCALE, nsplit=nsplit).float(), want)
        assert splits_of(cache._partials[(len(lens), n_kv, nsplit)], n_kv) >= least


@pytest.mark.parametrize("lens,n_kv,nsplit,least", CASES)
def test_paged_pool(lens, n_kv, nsplit, least):
    dev = require_gpu()
    gen = torch.Generator(device=dev).manual_seed(len(lens) + 1)
    layer, pool, bt, sl = ragged._paged(lens, n_kv, gen, dev)
    q = _queries(lens, n_kv, gen, dev)
    want = torch.cat([layer.attention(q[i:i + 1], pool, bt[i:i + 1], sl[i:i + 1], 7) for i in range(len(lens))]).float()
    for _ in range(2):
        assert_rows_close(layer.attention(q, pool, bt, sl, nsplit).float(), want)
        assert splits_of(layer._ws[(len(lens), n_kv, nsplit)], n_kv) >= least
    layer.check()
