"""Paged rows of few heads in all, which get one round of eight-wave blocks: both sides of the rule's lines, and pools of raw tiles, which two waves of such a block share."""
import numpy as np
import pytest
import torch

import test_gpu_ragged_rows as ragged
from common import assert_rows_close
from gpu_util import require_gpu
from test_gpu_long_row import splits_of

pytestmark = pytest.mark.gpu


def _even(n, lo, hi): return [lo + (hi - lo) * ((5 * i + 2) % n) // max(n - 1, 1) for i in range(n)]


# lengths, kv heads, splits asked for; splits of each row, if they are equal
CASES = [
    ([900] * 20, 2, 32, 6), ([900] * 40, 1, 32, 6),               # 40 heads on 240 CUs
    (_even(41, 200, 900), 1, 32, None),                             # 246 CUs
    ([2600] * 8, 8, 32, 4), (_even(8, 200, 3000), 8, 32, None),     # 64 heads
    ([10240, 100], 32, 32, None), ([10241, 100], 32, 32, None),     # 640 tiles, 641
    (_even(5, 1, 700), 13, 32, None),                               # 65 heads
    ([100, 2560, 900], 8, 32, None), ([100, 2561, 900], 8, 32, None), ([2561] * 3, 8, 32, 10), ([0, 1, 2600], 8, 11, None),     # ten splits: 160 tiles, 161 and more are planned
    ([500] * 5 + [20000], 4, 85, None), ([0, 5000, 3], 4, 64, None), ([16] * 2, 1, 200, 128),
]


@pytest.mark.parametrize("lens,n_kv,nsplit,each", CASES)
def test_rows(lens, n_kv, nsplit, each):
    dev = require_gpu()
    gen = torch.Generator(device=dev).manual_seed(len(lens) + nsplit)
    layer, pool, bt, sl = ragged._paged(lens, n_kv, gen, dev)
    q = torch.randn(len(lens), n_kv, 128, generator=gen, device=dev).to(torch.bfloat16)
    want = torch.cat([layer.attention(q[i:i + 1], pool, bt[i:i + 1], sl[i:i + 1], 7) for i in range(len(lens))]).float()
    for _ in range(3): assert_rows_close(layer.attention(q, pool, bt, sl, nsplit).float(), want)
    if each and lens[0] > 16 * each:
        q[0] = 0
        layer.attention(q, pool, bt, sl, nsplit)
        assert splits_of(layer._ws[(len(lens), n_kv, nsplit)], n_kv) == each
    layer.check()


@pytest.mark.parametrize("lens,n_kv,G", [([17], 1, 16), ([5000], 2, 4), (_even(8, 30, 900), 8, 2), (_even(3, 1, 400), 5, 7)])
@pytest.mark.parametrize("kinds", ["k", "v", "kv"])
def test_raw_tiles(lens, n_kv, G, kinds):
    """Bases that fit nothing on the sides `kinds`: each tile has one raw side or two.  Against attention over the same rows where all of them are compressed."""
    dev = require_gpu()
    from gaac_amd.codec import bases_from_hist, exponent_hist
    from gaac_amd.paged import BLOCK, LayerState, build_store_entries
    gen = torch.Generator(device=dev).manual_seed(len(lens) + n_kv)
    rows = [(ragged._rows(gen, L, n_kv, dev), ragged._rows(gen, L, n_kv, dev)) for L in lens]
    good, none = bases_from_hist(exponent_hist(ragged._rows(gen, 512, n_kv, dev), n_kv), n_kv), (torch.zeros(n_kv, 128, dtype=torch.uint8, device=dev),) * 2
    blocks = [-(-L // BLOCK) for L in lens]
    at = np.cumsum([0] + blocks)
    q = torch.randn(len(lens), n_kv * G, 128, generator=gen, device=dev).to(torch.bfloat16)
    sl, outs = torch.tensor(lens, dtype=torch.int32, device=dev), []
    for bad in ("", kinds):
        (k3, k4), (v3, v4) = none if "k" in bad else good, none if "v" in bad else good
        layer = LayerState(sum(blocks), n_kv, 2 * n_kv * sum(blocks), dict(k3=k3, k4=k4, v3=v3, v4=v4), device=dev)
        pool, bt = torch.zeros(LayerState.pool_bytes(sum(blocks), n_kv), dtype=torch.uint8, device=dev), np.zeros((len(lens), max(blocks)), np.int32)
        for i, (k, v) in enumerate(rows):
            bt[i, :blocks[i]] = np.arange(at[i], at[i + 1])
            layer.store(k, v, pool, torch.from_numpy(build_store_entries([0], [lens[i]], [bt[i]])).to(dev))
        if bad: assert int((layer.mt < 0).sum()) >= n_kv * len(bad) * sum(blocks)
        outs.append([layer.attention(q, pool, torch.from_numpy(bt).to(dev), sl, n).float() for n in (1, 3, 64)])
        layer.check()
    for got in outs[0] + outs[1]: assert_rows_close(got, outs[0][0])


# raw tiles among 1200 of a split: none, one, two of one thread of the block (512 apart) and of two, in the first 1024 tiles and in those behind them
@pytest.mark.parametrize("raw", [(), (5,), (5, 517), (5, 6), (5, 6, 7), (1030,), (1030, 1031), (5, 1100), (5, 1100, 1101), (5, 6, 1100), (0, 1023, 1024, 1198)])
@pytest.mark.parametrize("G", [2, 6])
def test_counts_of_raw_tiles(raw, G):
    dev = require_gpu()
    from gaac_amd.codec import bases_from_hist, exponent_hist
    from gaac_amd.paged import LayerState, build_store_entries
    gen = torch.Generator(device=dev).manual_seed(G + sum(raw))
    n, L = 1200, 1200 * 16
    k, v = (torch.randn(L, 1, 128, generator=gen, device=dev) for _ in range(2))
    for t in raw:      # exponents all over: escapes beyond a slot's room
        for x in (k, v): x[16 * t:16 * t + 16] *= torch.exp2(torch.randint(-24, 5, (16, 1, 128), generator=gen, device=dev).float())
    k, v = k.to(torch.bfloat16), v.to(torch.bfloat16)
    b3, b4 = bases_from_hist(exponent_hist(k, 1), 1)
    layer = LayerState(n, 1, 2 * n, dict(k3=b3, k4=b4, v3=b3, v4=b4), device=dev)
    pool, bt = torch.zeros(LayerState.pool_bytes(n, 1), dtype=torch.uint8, device=dev), np.arange(n, dtype=np.int32).reshape(1, n)
    layer.store(k, v, pool, torch.from_numpy(build_store_entries([0], [L], bt)).to(dev))
    assert (layer.mt < 0).nonzero().flatten().tolist() == [2 * t + j for t in raw for j in range(2)]
    q = (torch.randn(1, G, 128, generator=gen, device=dev) * 0.5).to(torch.bfloat16)
    p = torch.softmax(q[0].double() @ k[:, 0].double().T * 128 ** -0.5, -1)
    want = (p @ v[:, 0].double()).float()[None]
    for nsplit in (1, 2): assert_rows_close(layer.attention(q, pool, torch.from_numpy(bt).to(dev), torch.tensor([L], dtype=torch.int32, device=dev), nsplit).float().view(1, G, 128), want)
    layer.check()
