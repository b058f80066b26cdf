"""Launches that share their blocks out by the rows' lengths, against the same rows launched one at a time: one round and several, blocks
left over, rows that are empty, padded or a thousand times longer than the others, more rows than a wave has lanes and than are planned
for, over the slot cache and the paged pool, repeatedly on one workspace and under graph replay."""
import numpy as np
import pytest
import torch

from gpu_util import require_gpu

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


def _bound(want):
    """Each side rounds its softmax weights and its output to bf16 (half a unit, 2^-9, each): 2^-8 (sum p |v| + |out|) between two of them,
    with sum p |v| about 0.8 for unit Gaussian values under spread weights and |out| under concentrated ones."""
    return 2.0 ** -7 * max(want.abs().max().item(), 1.0)


def _rows(gen, n, n_kv, dev):
    return torch.randn(n, n_kv, 128, generator=gen, device=dev).to(torch.bfloat16)


CASES = [  # lengths, kv heads, query heads per kv head, splits
    ([700, 33], 2, 4, 5),
    ([5000] + [40] * 7, 8, 1, 16),                              # eight-wave blocks up to 256, most of them left over
    ([300 + 170 * i for i in range(32)], 8, 4, 2),             # one round of four-wave blocks
    ([300 + 170 * i for i in range(32)], 8, 4, 9),
    ([20000, 1, 16, 0, 17, 4000], 4, 5, 40),                   # an empty row
    ([9000 + 500 * (i % 5) for i in range(16)], 16, 2, 4),     # several rounds: every row takes its four splits
    ([16 * (i % 7) + 40 for i in range(70)], 2, 2, 3),         # more rows than a wave has lanes
    ([16 * (i % 5) + 20 for i in range(260)], 1, 16, 2),       # more rows than are planned for
]


@pytest.mark.parametrize("lens,n_kv,G,nsplit", CASES)
def test_slot_cache(lens, n_kv, G, nsplit):
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    gen = torch.Generator(device=dev).manual_seed(len(lens))
    B, n_q = len(lens), n_kv * G
    cache = CompressedKVCache(B, n_kv, max(lens) + 16, device=dev)
    for i, L in enumerate(lens):
        cache.prefill(i, _rows(gen, L, n_kv, dev), _rows(gen, L, n_kv, dev))
    slots = torch.randperm(B, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(dev)
    slots[B // 2] = -1
    q = (torch.randn(B, n_q, 128, generator=gen, device=dev) * 0.5).to(torch.bfloat16)
    want = torch.cat([cache.attention(q[i:i + 1], slots[i:i + 1], SCALE, nsplit=7) for i in range(B)]).float()
    for rnd in range(3):
        got = cache.attention(q, slots, SCALE, nsplit=nsplit).float()
        assert (got[B // 2] == 0).all()
        assert torch.isfinite(got).all() and (got - want).abs().max().item() <= _bound(want), rnd
        ws = cache._partials[(B, n_q, nsplit)]
        assert int(ws.epoch[0]) == rnd + 1 and ws.failure_bits() == 0
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = cache.attention(q, slots, SCALE, nsplit=nsplit)
    for _ in range(3):
        out.zero_(); g.replay(); torch.cuda.synchronize()
        assert (out.float() - want).abs().max().item() <= _bound(want)
    cache.check_capacity()


@pytest.mark.parametrize("lens,n_kv,G,nsplit", CASES)
def test_paged_pool(lens, n_kv, G, nsplit):
    dev = require_gpu()
    from gaac_amd.codec import bases_from_hist, exponent_hist
    from gaac_amd.paged import BLOCK, LayerState, build_store_entries
    gen = torch.Generator(device=dev).manual_seed(len(lens) + 1)
    B, n_q = len(lens), n_kv * G
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
    bt, sl = torch.from_numpy(bt).to(dev), torch.tensor(lens, dtype=torch.int32, device=dev)
    q = (torch.randn(B, n_q, 128, generator=gen, device=dev) * 0.5).to(torch.bfloat16)
    want = torch.cat([layer.attention(q[i:i + 1], pool, bt[i:i + 1], sl[i:i + 1], 7) for i in range(B)]).float()
    for rnd in range(3):
        got = layer.attention(q, pool, bt, sl, nsplit).float()
        assert torch.isfinite(got).all() and (got - want).abs().max().item() <= _bound(want), rnd
    layer.check()
