"""Split counts that a launch takes from its lengths, and merges of more half heads than merging blocks, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import gaac_oracle as O
from common import to_bf16, to_u16, randn_bf16, attention_error_bound
from gpu_util import require_gpu
from test_gpu_attention import _pages, _ref, SCALE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 16, 63, 64, 65, 129, 1000])      # around one split of four tiles, two, sixteen
@pytest.mark.parametrize("B,n_kv,G", [(1, 8, 4), (3, 2, 16)])
def test_splits_of_a_known_length(S, B, n_kv, G):
    dev = require_gpu()
    from gaac_amd import attention
    k16, v16, kp, vp = _pages(B, n_kv, S, dev, seed=21, soft=True)
    q16 = randn_bf16((B, n_kv * G, 128), seed=22)
    ref = _ref(q16, k16, v16, B, n_kv)
    for nsplit in (1, 2, 5, 31, 100, 2):
        got = O.bf16_to_f32(to_u16(attention(to_bf16(q16, dev), kp, vp, SCALE, nsplit=nsplit)))
        assert np.abs(got - ref).max() <= 2e-2 * np.abs(ref).max() + 1e-3, nsplit      # the bound of test_attention_matches_reference


@pytest.mark.parametrize("n_kv,G", [(1, 16), (2, 9), (1, 8)])
@pytest.mark.parametrize("L", [37, 1100])      # with empty splits, without
def test_more_half_heads_than_mergers(n_kv, G, L):
    """Nine query heads and up: the halves of an eight-wave block take a half head each, up to 32 splits in one round of records, then in more."""
    from gaac_amd import CompressedKVCache
    dev = require_gpu()
    cache = CompressedKVCache(1, n_kv, 1200, None, device=dev)
    k, v, q = randn_bf16((L, n_kv, 128), seed=31), randn_bf16((L, n_kv, 128), seed=32), randn_bf16((1, n_kv * G, 128), seed=33)
    cache.prefill(0, to_bf16(k, dev), to_bf16(v, dev))
    ref, tol = attention_error_bound(q[0], k, v, SCALE)
    slots = torch.zeros(1, dtype=torch.int32, device=dev)
    for nsplit in (15, 16, 17, 31, 32, 33, 63, 64, 65, 128, 300, 17):      # 300: four-wave blocks
        got = O.bf16_to_f32(to_u16(cache.attention(to_bf16(q, dev), slots, SCALE, nsplit=nsplit)))[0]
        assert (np.abs(got - ref) <= tol).all(), nsplit
    cache.check_capacity()


def test_max_len_of_any_kind_of_number():
    """launch_nsplit keeps its results: a zero-dimensional array or tensor, which changes in place or has no hash, is looked at in each call."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    from gaac_amd.kernel import launch_nsplit
    cache = CompressedKVCache(2, 8, 4096)
    slots, q = torch.arange(2, dtype=torch.int32, device=dev), torch.zeros(2, 8, 128, dtype=torch.bfloat16, device=dev)
    m, t = np.array(4000), torch.tensor(4000, device=dev)
    for n in (4000, 200, 1000):
        m[()] = n
        t.fill_(n)
        for given in (m, t, np.int64(n), n):
            cache._partials.clear()
            cache.attention(q, slots, 1.0, max_len=given)
            assert list(cache._partials) == [(2, 8, launch_nsplit(2, 8, n, True))]
