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
