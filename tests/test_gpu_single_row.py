"""A batch of one row: no more splits than fill one round of eight-wave blocks, whatever the caller asks for, and the results of a few splits."""
import pytest
import torch

import test_gpu_ragged_rows as ragged
from common import assert_rows_close
from gpu_util import require_gpu
from test_gpu_long_row import splits_of

pytestmark = pytest.mark.gpu

# tokens, kv heads, splits asked for
CASES = [(5000, 1, 256), (5000, 3, 256), (9001, 8, 32), (9001, 8, 33), (9001, 8, 256), (700, 130, 2), (700, 130, 5), (300, 300, 3), (1, 8, 64)]


@pytest.mark.parametrize("L,n_kv,nsplit", CASES)
def test_slot_cache(L, n_kv, nsplit):
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    gen = torch.Generator(device=dev).manual_seed(L + nsplit)
    cache = CompressedKVCache(2, n_kv, L + 16, device=dev)
    cache.prefill(1, ragged._rows(gen, L, n_kv, dev), ragged._rows(gen, L, n_kv, dev))
    slots = torch.ones(1, dtype=torch.int32, device=dev)
    q, zero = torch.randn(1, n_kv, 128, generator=gen, device=dev).to(torch.bfloat16), torch.zeros(1, n_kv, 128, dtype=torch.bfloat16, device=dev)
    want = cache.attention(q, slots, ragged.SCALE, nsplit=1).float()
    for _ in range(2): assert_rows_close(cache.attention(q, slots, ragged.SCALE, nsplit=nsplit).float(), want)
    cache.attention(zero, slots, ragged.SCALE, nsplit=nsplit)
    if 256 // n_kv > 1: assert splits_of(cache._partials[(1, n_kv, nsplit)], n_kv) <= 256 // n_kv      # (a single split leaves no records)


# wide: blocks per row that the block table has room for; a split is never planned longer than the 1024 tiles that are looked up at a time
@pytest.mark.parametrize("L,n_kv,nsplit,wide", [(*c, 0) for c in CASES] + [(9001, 32, 64, 10000), (20000, 64, 64, 70000)])
def test_paged_pool(L, n_kv, nsplit, wide):
    dev = require_gpu()
    gen = torch.Generator(device=dev).manual_seed(L + nsplit + 1)
    layer, pool, bt, sl = ragged._paged([L], n_kv, gen, dev)
    if wide: bt = torch.cat([bt, torch.zeros(1, wide - bt.shape[1], dtype=bt.dtype, device=dev)], dim=1).contiguous()
    q, zero = torch.randn(1, n_kv, 128, generator=gen, device=dev).to(torch.bfloat16), torch.zeros(1, n_kv, 128, dtype=torch.bfloat16, device=dev)
    want = layer.attention(q, pool, bt, sl, 1).float()
    for _ in range(2): assert_rows_close(layer.attention(q, pool, bt, sl, nsplit).float(), want)
    layer.attention(zero, pool, bt, sl, nsplit)
    most = max(256 // n_kv, -(-bt.shape[1] // 1024))
    if most > 1: assert splits_of(layer._ws[(1, n_kv, nsplit)], n_kv) <= most
    layer.check()


# tokens, kv heads, splits asked for, splits that the row gets: more heads than half the chip's CUs, where 256 / n_kv is one split
@pytest.mark.parametrize("L,n_kv,nsplit,want", [
    (2048, 128, 7, 2), (2048, 129, 7, 3), (2048, 170, 7, 3), (2049, 171, 7, 2), (2049, 256, 7, 2),      # up to 2048 tokens one split if it is not three
    (10240, 131, 9, 3), (10241, 131, 9, 9), (10241, 150, 9, 3),                                          # from 10241 on a round that is nearly full, or as asked
    (10240, 190, 9, 2), (10241, 223, 9, 9), (10241, 224, 9, 2), (2049, 257, 4, 4), (2049, 383, 4, 4), (2049, 520, 3, 3), (3000, 140, 2, 2)])
def test_many_heads(L, n_kv, nsplit, want):
    dev = require_gpu()
    gen = torch.Generator(device=dev).manual_seed(L + n_kv)
    layer, pool, bt, sl = ragged._paged([L], n_kv, gen, dev)
    q, zero = torch.randn(1, n_kv, 128, generator=gen, device=dev).to(torch.bfloat16), torch.zeros(1, n_kv, 128, dtype=torch.bfloat16, device=dev)
    ref = layer.attention(q, pool, bt, sl, 1).float()
    assert_rows_close(layer.attention(q, pool, bt, sl, nsplit).float(), ref)
    layer.attention(zero, pool, bt, sl, nsplit)
    ws = layer._ws[(1, n_kv, nsplit)]
    assert int(ws.epoch[0]) == 2 and splits_of(ws, n_kv) == want      # (a launch of one split leaves the records, all zero, and the epoch alone)
    layer.check()


@pytest.mark.parametrize("L,n_kv,nsplit", [(2048, 171, 7), (2048, 300, 7), (2049, 384, 4), (10240, 500, 4), (700, 130, 2)])
def test_many_heads_in_one_split(L, n_kv, nsplit):
    """A single split is the result: no record is left."""
    dev = require_gpu()
    gen = torch.Generator(device=dev).manual_seed(L + n_kv)
    layer, pool, bt, sl = ragged._paged([L], n_kv, gen, dev)
    q = torch.randn(1, n_kv, 128, generator=gen, device=dev).to(torch.bfloat16)
    ref = layer.attention(q, pool, bt, sl, 1).float()
    assert_rows_close(layer.attention(q, pool, bt, sl, nsplit).float(), ref)
    assert not layer._ws[(1, n_kv, nsplit)].pm.any()
    layer.check()
