"""Launches that share their blocks out by the rows' lengths, against the same rows launched one at a time: one round and several, blocks
left over, rows that are empty, padded or a thousand times longer than the others, more rows than a wave has lanes and than are planned
for, over the slot cache and the paged pool, repeatedly on one workspace and under graph replay."""
import numpy as np
import pytest
import torch

from common import assert_rows_close
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


def _rows(gen, n, n_kv, dev):
    return torch.randn(n, n_kv, 128, generator=gen, device=dev).to(torch.bfloat16)


# lengths, kv heads, query heads per kv head, splits, and what the launch is to do with them: NSPLIT splits for every row, rows SHARED out
# over one round, or a number: that many splits for every row
NSPLIT, SHARED = "nsplit", "shared"
CASES = [
    ([700, 33], 2, 4, 5, NSPLIT),                                        # few blocks, short splits: not planned
    ([12000, 700, 3000, 40], 8, 1, 8, SHARED),                          # eight-wave blocks
    ([12000, 11900, 11800, 11950], 8, 1, 8, NSPLIT),                    # eight-wave blocks, rows within 1/32 of each other
    ([5000] + [40] * 7, 8, 1, 16, SHARED),                              # four-wave blocks, most of them left over
    ([300 + 170 * i for i in range(32)], 8, 4, 2, SHARED),             # all of them resident
    ([300 + 170 * i for i in range(32)], 8, 4, 9, SHARED),
    ([20000, 1, 16, 0, 17, 4000], 4, 5, 40, SHARED),                    # an empty row
    ([9000 + 500 * (i % 5) for i in range(16)], 16, 2, 4, NSPLIT),     # several rounds, longest first, equal lengths among them
    ([3000] * 20, 16, 2, 4, NSPLIT),                                    # equal rows, several rounds
    ([6400] * 24, 8, 1, 3, 2),                                          # one round, instead of one and a nearly empty one
    ([1000] * 9, 8, 2, 8, 7),                                           # equal rows, one round
    ([1000] * 40, 8, 1, 4, 1),
    ([16 * (i % 7) + 40 for i in range(70)], 2, 2, 3, SHARED),         # more rows than a wave has lanes
    ([100 + 40 * (i // 3) for i in range(130)], 2, 2, 3, SHARED),
    ([100 + 40 * (i // 3) for i in range(130)], 4, 2, 1, NSPLIT),      # order only
    ([100 + 120 * (i // 3) for i in range(130)], 5, 1, 2, NSPLIT),
    ([600] * 130, 2, 2, 3, 1),
    ([16 * (i % 5) + 20 for i in range(256)], 1, 16, 2, SHARED),       # as many rows as are planned for
    ([16 * (i % 5) + 20 for i in range(260)], 1, 16, 2, NSPLIT),       # and more
]


def _check_splits(ws, B, n_q, nsplit, expect):
    """The records that the workspace's first launch left: one per query head and split of the rows with more than one split."""
    n = int(((ws.pm >> 32) == 1).sum())
    if nsplit == 1: assert n == 0
    elif expect == SHARED: assert n != B * n_q * nsplit
    else:
        ns = nsplit if expect == NSPLIT else expect
        assert n == (B * n_q * ns if ns > 1 else 0)


@pytest.mark.parametrize("lens,n_kv,G,nsplit,expect", CASES)
def test_slot_cache(lens, n_kv, G, nsplit, expect):
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    gen = torch.Generator(device=dev).manual_seed(len(lens))
    B, n_q = len(lens), n_kv * G
    cache = CompressedKVCache(B, n_kv, max(lens) + 16, device=dev)
    for i, L in enumerate(lens):
        cache.prefill(i, _rows(gen, L, n_kv, dev), _rows(gen, L, n_kv, dev))
    slots = torch.randperm(B, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(dev)
    padded = B // 2 if len(set(lens)) > 1 and max(lens) > 1.1 * min(lens) else None      # a padded row where it leaves the lengths as unequal as they were
    if padded is not None: slots[padded] = -1
    q = (torch.randn(B, n_q, 128, generator=gen, device=dev) * 0.5).to(torch.bfloat16)
    want = torch.cat([cache.attention(q[i:i + 1], slots[i:i + 1], SCALE, nsplit=7) for i in range(B)]).float()
    for rnd in range(3):
        got = cache.attention(q, slots, SCALE, nsplit=nsplit).float()
        assert padded is None or (got[padded] == 0).all()
        assert_rows_close(got, want)
        ws = cache._partials[(B, n_q, nsplit)]
        if rnd == 0: _check_splits(ws, B, n_q, nsplit, expect)
        assert int(ws.epoch[0]) == (rnd + 1 if nsplit > 1 else 0) and ws.failure_bits() == 0
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = cache.attention(q, slots, SCALE, nsplit=nsplit)
    for _ in range(3):
        out.zero_(); g.replay(); torch.cuda.synchronize()
        assert_rows_close(out.float(), want)
    cache.check_capacity()


def _paged(lens, n_kv, gen, dev):
    """(layer, pool, block table, lengths) with the rows stored in permuted blocks."""
    from gaac_amd.codec import bases_from_hist, exponent_hist
    from gaac_amd.paged import BLOCK, LayerState, build_store_entries
    B = len(lens)
    n_blk = [-(-L // BLOCK) for L in lens]
    perm = np.random.default_rng(3).permutation(sum(n_blk)).astype(np.int32)
    at = np.cumsum([0] + n_blk)
    bt = np.zeros((B, max(n_blk)), np.int32)
    b3, b4 = bases_from_hist(exponent_hist(_rows(gen, 512, n_kv, dev), n_kv), n_kv)
    layer = LayerState(sum(n_blk), n_kv, 2 * n_kv * (B + 8), dict(k3=b3, k4=b4, v3=b3, v4=b4), device=dev)
    pool = torch.zeros(LayerState.pool_bytes(sum(n_blk), n_kv), dtype=torch.uint8, device=dev)
    for i, L in enumerate(lens):
        bt[i, :n_blk[i]] = perm[at[i]:at[i + 1]]
        if L: layer.store(_rows(gen, L, n_kv, dev), _rows(gen, L, n_kv, dev), pool, torch.from_numpy(build_store_entries([0], [L], [bt[i]])).to(dev))
    return layer, pool, torch.from_numpy(bt).to(dev), torch.tensor(lens, dtype=torch.int32, device=dev)


@pytest.mark.parametrize("lens,n_kv,G,nsplit,expect", CASES)
def test_paged_pool(lens, n_kv, G, nsplit, expect):
    dev = require_gpu()
    gen = torch.Generator(device=dev).manual_seed(len(lens) + 1)
    B, n_q = len(lens), n_kv * G
    layer, pool, bt, sl = _paged(lens, n_kv, gen, dev)
    q = (torch.randn(B, n_q, 128, generator=gen, device=dev) * 0.5).to(torch.bfloat16)
    want = torch.cat([layer.attention(q[i:i + 1], pool, bt[i:i + 1], sl[i:i + 1], 7) for i in range(B)]).float()
    for rnd in range(3):
        got = layer.attention(q, pool, bt, sl, nsplit).float()
        assert_rows_close(got, want)
        if rnd == 0: _check_splits(layer._ws[(B, n_q, nsplit)], B, n_q, nsplit, expect)
    layer.check()


def test_rows_of_many_heads_go_longest_first():
    """No limit on rows x heads: the first records are those of the longest row, wherever it stands in the batch (the largest score of a
    split does not depend on the order of its tiles)."""
    dev = require_gpu()
    gen = torch.Generator(device=dev).manual_seed(5)
    lens, n_kv = [100] * 40 + [34000] + [50] * 29, 60
    layer, pool, bt, sl = _paged(lens, n_kv, gen, dev)
    q = torch.randn(len(lens), n_kv, 128, generator=gen, device=dev).to(torch.bfloat16)
    want = layer.attention(q[40:41], pool, bt[40:41], sl[40:41], 2).float()
    got = layer.attention(q, pool, bt, sl, 2).float()
    assert_rows_close(got[40:41], want)
    first, alone = layer._ws[(len(lens), n_kv, 2)].pm[:2 * n_kv], layer._ws[(1, n_kv, 2)].pm
    assert torch.equal(first & 0xFFFFFFFF, alone & 0xFFFFFFFF)
    layer.check()


def test_the_last_block_waits_for_a_long_launch():
    """A row of sixteen million tokens next to one of a single token, four blocks in all: the grid's last block is done at once and waits
    for the others for a good part of a second before it advances the epoch."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    gen = torch.Generator(device=dev).manual_seed(9)
    b = torch.full((1, 128), 120, dtype=torch.uint8)
    cache = CompressedKVCache(2, 1, 1 << 24, dict(k3=b, k4=b, v3=b, v4=b), device=dev)
    part = 1 << 16
    k, v = (_rows(gen, part, 1, dev).repeat(255, 1, 1) for _ in range(2))
    cache.prefill(0, k, v)
    cache.prefill(1, k[:1], v[:1])
    del k, v
    q = (torch.randn(2, 1, 128, generator=gen, device=dev) * 0.5).to(torch.bfloat16)
    slots = torch.arange(2, dtype=torch.int32, device=dev)
    want = cache.attention(q, slots, SCALE, nsplit=64).float()
    for rnd in range(2):
        assert_rows_close(cache.attention(q, slots, SCALE, nsplit=2).float(), want)
        ws = cache._partials[(2, 1, 2)]
        assert ws.failure_bits() == 0 and int(ws.epoch[0]) == rnd + 1
    cache.check_capacity()
