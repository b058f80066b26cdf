"""CompressedKVCache.prefill at the edges of its launches: prompts shorter than a tile, whole tiles only, chunk borders of the exponent
histogram, prompts given as views of other layouts, windows that have to grow, windows that may not, and arguments it rejects."""
import numpy as np
import pytest
import torch

from oracle import gaac_oracle as O
from common import kv_like16, to_bf16, to_u16
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu
N_KV = 3


def _tokens(L, seed, outliers=1e-3):
    return np.ascontiguousarray(kv_like16(N_KV, L, seed=seed, outliers=outliers, scale_seed=7).transpose(1, 0, 2))


def _held(cache, slot, k16, v16):
    dk, dv = cache.decompress(slot)
    return np.array_equal(to_u16(dk), k16) and np.array_equal(to_u16(dv), v16)


@pytest.mark.parametrize("L", [1, 15, 16, 17, 255, 256, 257, 511 * 16, 2000])
def test_calibrated_prompts_equal_the_oracle(L):
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    cache = CompressedKVCache(3, N_KV, L + 40, device=dev)
    k16, v16 = _tokens(L, L), _tokens(L, L + 1)
    other = _tokens(min(L, 40), 3)
    cache.prefill(0, to_bf16(other, dev), to_bf16(other, dev))
    cache.prefill(1, to_bf16(k16, dev), to_bf16(v16, dev))
    for st, x16 in ((cache.k, k16), (cache.v, v16)):
        b3, b4 = O.bases_from_hist(O.exponent_hist(x16, N_KV), N_KV)
        assert np.array_equal(st.base3[N_KV:2 * N_KV].cpu().numpy(), b3) and np.array_equal(st.base4[N_KV:2 * N_KV].cpu().numpy(), b4)
    assert cache.S.tolist()[N_KV:2 * N_KV] == [L // 16 * 16] * N_KV and cache.tail_len.tolist()[N_KV:2 * N_KV] == [L % 16] * N_KV
    assert cache.S.tolist()[2 * N_KV:] == [0] * N_KV
    assert _held(cache, 1, k16, v16) and _held(cache, 0, other, other)
    if L >= 16:
        page = O.encode(np.ascontiguousarray(k16[:L // 16 * 16].transpose(1, 0, 2)), "k", cache.k.base3[N_KV:2 * N_KV].cpu().numpy(), cache.k.base4[N_KV:2 * N_KV].cpu().numpy(), N_KV)
        assert np.array_equal(cache.k.ovf_used[N_KV:2 * N_KV].cpu().numpy(), np.diff(page.ovf_head_start))
        assert np.array_equal(cache.k.tile_off[N_KV:2 * N_KV, :L // 16].cpu().numpy(), page.tile_off)


def test_empty_prompt_clears_the_slot():
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    cache = CompressedKVCache(1, N_KV, 64, device=dev)
    x = to_bf16(_tokens(40, 1), dev)
    cache.prefill(0, x, x)
    cache.prefill(0, x[:0], x[:0])
    assert not cache.S.any() and not cache.tail_len.any() and not cache.k.ovf_used.any()


def test_views_of_other_layouts():
    """Slices of a fused qkv projection (row stride wider than the heads), a head-major tensor seen token-major, a misaligned slice."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    L = 213
    k16, v16 = _tokens(L, 11), _tokens(L, 12)
    qkv = torch.zeros(L, 4 + 2 * N_KV, 128, dtype=torch.bfloat16, device=dev)
    qkv[:, 4:4 + N_KV] = to_bf16(k16, dev); qkv[:, 4 + N_KV:] = to_bf16(v16, dev)
    major = to_bf16(np.ascontiguousarray(v16.transpose(1, 0, 2)), dev).transpose(0, 1)
    odd = torch.zeros(L * N_KV * 128 + 1, dtype=torch.bfloat16, device=dev)[1:].view(L, N_KV, 128)
    odd.copy_(to_bf16(k16, dev))
    cache = CompressedKVCache(3, N_KV, 256, device=dev)
    cache.prefill(0, qkv[:, 4:4 + N_KV], qkv[:, 4 + N_KV:])
    cache.prefill(1, qkv[:, 4:4 + N_KV], major)
    cache.prefill(2, odd, major)
    assert all(_held(cache, s, k16, v16) for s in range(3))


def test_windows_grow_for_a_prompt_and_refuse_when_they_may_not():
    """Mostly raw groups: about 1000 escape bytes a tile against windows of 16."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    L = 330
    k16, v16, small = _tokens(L, 21, outliers=0.3), _tokens(L, 22), _tokens(30, 23)
    cache = CompressedKVCache(2, N_KV, 512, ovf_bytes_per_tile=64, device=dev)
    cache.prefill(1, to_bf16(small, dev), to_bf16(small, dev))
    before = cache.k.ovf_cap
    cache.prefill(0, to_bf16(k16, dev), to_bf16(v16, dev))
    assert cache.k.ovf_cap == cache.v.ovf_cap > before
    assert int(cache.k.ovf_used.max()) + 1288 <= cache.k.ovf_cap
    assert _held(cache, 0, k16, v16) and _held(cache, 1, small, small)
    fixed = CompressedKVCache(2, N_KV, 512, ovf_bytes_per_tile=64, device=dev)
    fixed.growable = False
    fixed.prefill(1, to_bf16(small, dev), to_bf16(small, dev))
    with pytest.raises(RuntimeError, match="window must grow"):
        fixed.prefill(0, to_bf16(k16, dev), to_bf16(v16, dev))
    assert fixed.S.tolist()[:N_KV] == [0] * N_KV      # no head reads past its window
    assert _held(fixed, 1, small, small)


@pytest.mark.parametrize("raw_k,raw_v", [(0.0, 0.02), (0.02, 0.0), (0.02, 0.05), (0.05, 0.02), (0.0, 0.3), (0.3, 0.3)])
def test_windows_grow_for_k_then_for_v(raw_k, raw_v):
    """Short slots, whose default windows are smaller than the headroom, so that the first prompt makes them grow: for K's largest head,
    and again for V's only if it needs more than that gave.  The window size that results is part of the cache's layout."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    L = 73
    k16, v16 = _tokens(L, 31, outliers=raw_k), _tokens(L, 32, outliers=raw_v)
    cache = CompressedKVCache(2, N_KV, L + 7, device=dev)
    want = cache.k.ovf_cap
    cache.prefill(1, to_bf16(k16, dev), to_bf16(v16, dev))
    for st in (cache.k, cache.v):
        need = int(st.ovf_used.max()) + 1288
        if need > want: want = max(2 * want, need + 4096 + 7) // 8 * 8
    assert cache.k.ovf_cap == cache.v.ovf_cap == want
    assert cache.k.ovf.numel() == cache.v.ovf.numel() == 2 * N_KV * want
    assert cache.k.head_start.tolist() == cache.v.head_start.tolist() == [i * want for i in range(2 * N_KV + 1)]
    assert _held(cache, 1, k16, v16)


@pytest.mark.parametrize("calibrate", [True, False])
@pytest.mark.parametrize("L", [1, 15])
def test_prompts_shorter_than_a_tile_are_put_in_place_without_a_wait(L, calibrate):
    """They have no escapes to wait for: captured and replayed with new rows in the same buffers, and from other float types."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    b = torch.full((N_KV, 128), 120, dtype=torch.uint8)
    cache = CompressedKVCache(3, N_KV, 64, None if calibrate else dict(k3=b, k4=b, v3=b, v4=b), device=dev)
    k16, v16 = _tokens(L, 41), _tokens(L, 42)
    k, v = to_bf16(k16, dev), to_bf16(v16, dev)
    cache.prefill(0, k, v)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g): cache.prefill(1, k, v)
    for seed in (43, 44, 45):
        a16, c16 = _tokens(L, seed), _tokens(L, seed + 10)
        k.copy_(to_bf16(a16, dev)); v.copy_(to_bf16(c16, dev))
        g.replay(); torch.cuda.synchronize()
        assert _held(cache, 1, a16, c16) and _held(cache, 0, k16, v16)
        if calibrate: assert np.array_equal(cache.k.base3[N_KV:2 * N_KV].cpu().numpy(), O.bases_from_hist(O.exponent_hist(a16, N_KV), N_KV)[0])
    cache.prefill(2, to_bf16(k16, dev).float(), to_bf16(v16, dev).float())
    assert _held(cache, 2, k16, v16)
    if not calibrate:
        cache.prefill(2, to_bf16(v16, "cpu"), to_bf16(k16, "cpu").double())
        assert _held(cache, 2, v16, k16)
    assert cache.S.tolist() == [0] * 3 * N_KV and cache.tail_len.tolist() == [L] * 3 * N_KV


def test_rejected_arguments():
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    cache = CompressedKVCache(2, N_KV, 64, device=dev)
    x = to_bf16(_tokens(32, 1), dev)
    with pytest.raises(RuntimeError, match="slot"): cache.prefill(2, x, x)
    with pytest.raises(RuntimeError, match="prefill expects"): cache.prefill(0, x, x[:16])
    with pytest.raises(RuntimeError, match="prefill expects"): cache.prefill(0, x.float(), x.float())
    with pytest.raises(AssertionError): cache.prefill(0, x.repeat(3, 1, 1), x.repeat(3, 1, 1))
