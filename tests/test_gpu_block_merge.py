"""The merges at the end of a split launch where they change form: query heads to waves of a block (two waves a head, a wave a head, several heads a wave), one
split, more splits than a merging lane's first round of records (32 or 64) and than a wave has lanes, for blocks of eight waves and of four."""
import numpy as np
import pytest

from oracle import gaac_oracle as O
from common import to_bf16, to_u16, randn_bf16
from gpu_util import require_gpu
from test_gpu_attention import _pages, _ref, SCALE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_kv,G", [(1, 1), (1, 4), (1, 5), (1, 8), (1, 9), (1, 16), (8, 2), (8, 3), (8, 5), (8, 9)])      # 8 heads: blocks of four waves from 33 splits on
def test_merges(n_kv, G):
    dev = require_gpu()
    from gaac_amd import attention
    S = 5000      # 313 tiles: 79 splits of four
    k16, v16, kp, vp = _pages(1, n_kv, S, dev, seed=27, soft=True)
    q16 = randn_bf16((1, n_kv * G, 128), seed=28)
    ref = _ref(q16, k16, v16, 1, n_kv)
    for nsplit in (1, 33, 40, 79, 2):
        got = O.bf16_to_f32(to_u16(attention(to_bf16(q16, dev), kp, vp, SCALE, nsplit=nsplit)))
        assert np.abs(got - ref).max() <= 2e-2 * np.abs(ref).max() + 1e-3, nsplit      # the bound of test_attention_matches_reference
