"""The merge of heads with few splits, on both sides of the line between the wave-wise and the block-wise merge (at most sixteen
splits and fewer than half heads; up to eight and beyond in different registers), with empty splits among them and launches of both block shapes."""
import numpy as np
import pytest
import torch

from oracle import gaac_oracle as O
from common import to_bf16, to_u16, randn_bf16
from gpu_util import require_gpu
from test_gpu_attention import _pages, _ref, SCALE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,n_kv,G", [(1, 2, 1), (1, 3, 2), (2, 1, 5), (1, 2, 16), (5, 16, 5)])      # the last: four-wave blocks from four splits on
@pytest.mark.parametrize("S", [33, 700, 1000])      # 1000: sixteen splits of four tiles, none empty
def test_few_splits(B, n_kv, G, S):
    dev = require_gpu()
    from gaac_amd import attention
    k16, v16, kp, vp = _pages(B, n_kv, S, dev, seed=17, soft=True)
    q16 = randn_bf16((B, n_kv * G, 128), seed=18)
    ref = _ref(q16, k16, v16, B, n_kv)
    for nsplit in (2, 3, 7, 8, 9, 10, 15, 16, 17, 2):      # 2 again: on records that launches of other shapes have left
        got = O.bf16_to_f32(to_u16(attention(to_bf16(q16, dev), kp, vp, SCALE, nsplit=nsplit)))
        assert np.isfinite(got).all()
        assert np.abs(got - ref).max() <= 2e-2 * np.abs(ref).max() + 1e-3, nsplit      # the bound of test_attention_matches_reference
