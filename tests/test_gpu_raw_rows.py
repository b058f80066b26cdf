"""GPU tests of the rows that attention takes uncompressed: the raw tail of a cache head and the raw tiles of the paged pool (both sides raw, or
one decoded beside the other), against attention in 64 bits."""
import numpy as np
import pytest
import torch

from oracle import gaac_oracle as O
from common import to_bf16, to_u16, randn_bf16
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


def _ref64(q16, k16, v16):
    """Attention of q16 [n_q, 128] over k16, v16 [L, n_kv, 128] in float64, and per output the largest value that is summed."""
    G = q16.shape[0] // k16.shape[1]
    out, size = np.zeros(q16.shape), np.zeros(q16.shape)
    for j in range(q16.shape[0]):
        k, v = (O.bf16_to_f32(x[:, j // G]).astype(np.float64) for x in (k16, v16))
        s = k @ O.bf16_to_f32(q16[j]).astype(np.float64) * SCALE
        p = np.exp(s - s.max()); p /= p.sum()
        out[j], size[j] = p @ v, p @ np.abs(v)
    return out, size


@pytest.mark.parametrize("n_kv,G", [(1, 16), (8, 1), (2, 6)])
@pytest.mark.parametrize("L", [1, 3, 4, 5, 15])
def test_a_tail_alone_is_exact_to_32_bit_sums(n_kv, G, L):
    """Nothing but a tail: weights and sums stay in 32 bits, so what is left is the rounding of the output to bf16 (half a unit of its 8
    bits: up to 2^-8 of it) and some thirty roundings of 32-bit sums and an exponential of at most a few units (2^-19 of the summed
    values).  Rows behind the tail's last one hold Inf and NaN."""
    from gaac_amd import CompressedKVCache
    dev = require_gpu()
    cache = CompressedKVCache(2, n_kv, 64, None, device=dev)
    cache.k.tail.fill_(float("inf")); cache.v.tail.fill_(float("nan"))
    k, v, q = randn_bf16((L, n_kv, 128), seed=L), randn_bf16((L, n_kv, 128), seed=L + 50), randn_bf16((1, n_kv * G, 128), seed=7, scale=2.0)
    cache.prefill(1, to_bf16(k, dev), to_bf16(v, dev))
    slots = torch.tensor([1], dtype=torch.int32, device=dev)
    want, size = _ref64(q[0], k, v)
    for nsplit in (1, 3):
        got = O.bf16_to_f32(to_u16(cache.attention(to_bf16(q, dev), slots, SCALE, nsplit=nsplit)))[0]
        assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -19 * size).all()


@pytest.mark.parametrize("S,nsplit", [(48, 1), (48, 5), (64, 2), (50, 300)])
@pytest.mark.parametrize("far", ["k", "v", "kv"])
def test_half_raw_tiles_among_others(S, nsplit, far):
    """Finished tiles whose K, V or both sides stay raw (exponents far from the bases), several in a split, beside compressed ones and a block
    that is still filling."""
    from gaac_amd.paged import LayerState, build_store_entries
    dev = require_gpu()
    n_kv, G = 2, 5
    ones = torch.full((n_kv, 128), 120, dtype=torch.uint8)
    st = LayerState(8, n_kv, 40, dict(k3=ones, k4=ones - 4, v3=ones, v4=ones - 4), 32, dev)
    buf = torch.zeros(LayerState.pool_bytes(8, n_kv, 32), dtype=torch.uint8, device=dev)

    def rows(seed, raw):      # exponents 120..123; in odd tiles 100..103 where the side is to stay raw
        rng = np.random.default_rng(seed)
        e = rng.integers(120, 124, (S, n_kv, 128))
        if raw: e[(np.arange(S) // 16) % 2 == 1] = rng.integers(100, 104, (int(((np.arange(S) // 16) % 2 == 1).sum()), n_kv, 128))
        return (rng.integers(0, 2, e.shape) << 15 | e << 7 | rng.integers(0, 128, e.shape)).astype(np.uint16)
    k, v = rows(1, "k" in far), rows(2, "v" in far)
    table = np.array([5, 2, 7, 0], np.int32)
    st.store(to_bf16(k, dev), to_bf16(v, dev), buf, torch.from_numpy(build_store_entries([0], [S], [table])).to(dev))
    mt = st.mt.cpu().numpy().reshape(-1, n_kv, 2)[2] < 0
    assert mt[:, 0].all() == ("k" in far) and mt[:, 1].all() == ("v" in far)
    q = randn_bf16((1, n_kv * G, 128), seed=3)
    out = st.attention(to_bf16(q, dev), buf, torch.from_numpy(table).view(1, -1).to(dev), torch.tensor([S], dtype=torch.int32, device=dev), nsplit, max_seq_len=S)
    got = O.bf16_to_f32(to_u16(out)).reshape(n_kv * G, 128)
    want, size = _ref64(q[0], k, v)
    # weights of compressed tiles and the output are rounded to bf16, by up to 2^-8 each; the sums as in a tail alone
    assert (np.abs(got - want) <= 2.0 ** -8 * (np.abs(want) + size) + 2.0 ** -19 * size).all()
    st.check()


def test_raw_tiles_beyond_the_first_1024_of_a_split():
    """One split over 1100 tiles: the raw tiles of the second round (and the filling block) join those of the first."""
    from gaac_amd.paged import LayerState, build_store_entries
    dev = require_gpu()
    n_kv, G, S = 1, 2, 1100 * 16 + 5
    blocks = -(-S // 16)
    ones = torch.full((n_kv, 128), 118, dtype=torch.uint8)
    st = LayerState(blocks, n_kv, 64, dict(k3=ones, k4=ones - 4, v3=ones, v4=ones - 4), 16, dev)
    buf = torch.zeros(LayerState.pool_bytes(blocks, n_kv, 16), dtype=torch.uint8, device=dev)
    rng = np.random.default_rng(4)
    e = rng.integers(118, 125, (2, S, n_kv, 128))
    for side, t in ((0, 3), (1, 500), (0, 1030), (1, 1030), (1, 1090)): e[side, 16 * t:16 * t + 16] = rng.integers(126, 128, (16, n_kv, 128)) - 22 * (side == 0)
    k, v = (rng.integers(0, 2, e.shape) << 15 | e << 7 | rng.integers(0, 128, e.shape)).astype(np.uint16)
    table = rng.permutation(blocks).astype(np.int32)
    st.store(to_bf16(k, dev), to_bf16(v, dev), buf, torch.from_numpy(build_store_entries([0], [S], [table])).to(dev))
    assert int((st.mt < 0).sum()) == 5 + 2
    q = randn_bf16((1, n_kv * G, 128), seed=5)
    out = st.attention(to_bf16(q, dev), buf, torch.from_numpy(table).view(1, -1).to(dev), torch.tensor([S], dtype=torch.int32, device=dev), 1, max_seq_len=S)
    want, size = _ref64(q[0], k, v)
    assert (np.abs(O.bf16_to_f32(to_u16(out)).reshape(G, 128) - want) <= 2.0 ** -8 * (np.abs(want) + size) + 2.0 ** -19 * size).all()
