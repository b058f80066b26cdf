"""The tile encoder at the edges of the room its escape bytes have, and the tile decoder at every combination of tiers that a lane can hold (its four groups raw, 4-bit or 3-bit): what it reads of the escape bytes,
and where it takes them from, depends on that.  Pages and paged slots, rows of every alignment; the result is the input, bit for bit."""
import itertools
import numpy as np
import pytest
import torch

from common import to_bf16, to_u16
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu
B3, B4 = 120, 116      # bases: 3-bit groups hold exponents 120..127, 4-bit ones 116..131


def _tiers_to_rows(tiers, kind, rng):
    """uint16 [H, S, 128] whose groups (of stored order) have the given tiers [H, S, 16]: 0, 1 or 3."""
    from gaac_amd.codec import perm
    H, S, _ = tiers.shape
    e = rng.integers(120, 128, (H, S, 16, 8))
    e = np.where(tiers[..., None] == 1, rng.integers(116, 132, e.shape), e)
    e = np.where(tiers[..., None] == 3, rng.integers(0, 255, e.shape), e)
    first = e[..., 0]
    first[tiers == 1] = 131      # outside the three-bit window
    first[tiers == 3] = 20       # outside both
    x = (e.reshape(H, S, 128) << 7 | rng.integers(0, 128, (H, S, 128)) | rng.integers(0, 2, (H, S, 128)) << 15).astype(np.uint16)
    out = np.empty_like(x)
    out[..., perm(kind).numpy()] = x
    return out


def _case(kind, H, S, p_raw, seed):
    rng = np.random.default_rng(seed)
    tiers = rng.choice([0, 1, 3], (H, S, 16), p=[(1 - p_raw) / 2, (1 - p_raw) / 2, p_raw])
    return tiers, _tiers_to_rows(tiers, kind, rng)


def _lane_combinations(tiers, kind):
    t = tiers[:, :tiers.shape[1] // 16 * 16]
    lanes = t.reshape(-1, 4) if kind == "k" else t.reshape(t.shape[0], -1, 4, 16).transpose(0, 1, 3, 2).reshape(-1, 4)
    return {tuple(int(v) for v in r) for r in lanes}


@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("S,p_raw", [(1, 1.0), (17, 0.0), (333, 0.3), (160, 1.0)])
def test_pages_of_every_combination_of_tiers(kind, S, p_raw):
    dev = require_gpu()
    from gaac_amd import Codec, TileEncoder, _lib
    H = 3
    tiers, x16 = _case(kind, H, S, p_raw, seed=S)
    if p_raw == 0.3: assert _lane_combinations(tiers, kind) == set(itertools.product((0, 1, 3), repeat=4))
    full = lambda v: torch.full((H, 128), v, dtype=torch.uint8)
    page = TileEncoder(kind).encode(Codec(H).set_bases(full(B3), full(B4)), to_bf16(x16, dev))
    n = int(page.ovf_head_start[-1])
    assert n == int((tiers == 1).sum() + 5 * (tiers == 3).sum())
    assert np.array_equal(to_u16(Codec.decode(page)), x16)
    # a stream at every alignment, and rows that are not 16-byte aligned
    p = _lib.ptr
    for shift, stride in ((1, 128), (2, 132), (3, 129)):
        ovf = torch.full((n + 8 + shift,), 255, dtype=torch.uint8, device=dev)
        ovf[shift:shift + n] = page.ovf[:n]
        out = torch.zeros(H, S, stride, dtype=torch.bfloat16, device=dev)
        _lib.call("gaac_decode_tiles", int(kind == "v"), p(page.sm), p(page.codes), p(page.flags), p(page.tile_off), p(ovf[shift:]), p(page.ovf_head_start),
                  p(page.base3), p(page.base4), H, None, H, S, page.sm.shape[1] // 128, p(out), S * stride, stride, _lib.stream())
        got = to_u16(out)
        assert np.array_equal(got[..., :128], x16) and not got[..., 128:].any()


@pytest.mark.parametrize("ovf_slot,p_raw", [(144, 0.02), (1280, 0.5), (1280, 1.0)])
def test_paged_slots_of_every_combination_of_tiers(ovf_slot, p_raw):
    dev = require_gpu()
    from gaac_amd.paged import LayerState, build_store_entries
    n_kv, L = 2, 167
    k16, v16 = (_case(kind, n_kv, L, p_raw, seed=5)[1].transpose(1, 0, 2) for kind in "kv")
    k, v = to_bf16(np.ascontiguousarray(k16), dev), to_bf16(np.ascontiguousarray(v16), dev)
    full = lambda b: torch.full((n_kv, 128), b, dtype=torch.uint8)
    blocks = -(-L // 16)
    table = np.random.default_rng(1).permutation(blocks).astype(np.int32)
    layer = LayerState(blocks, n_kv, blocks * 2 * n_kv, dict(k3=full(B3), k4=full(B4), v3=full(B3), v4=full(B4)), ovf_slot=ovf_slot)
    pool = torch.full((LayerState.pool_bytes(blocks, n_kv, ovf_slot),), 255, dtype=torch.uint8, device=dev)
    layer.store(k, v, pool, torch.from_numpy(build_store_entries([0], [L], [table])).to(dev))
    pairs = torch.tensor([(int(b), 16 * i, min(16, L - 16 * i)) for i, b in enumerate(table)], dtype=torch.int32, device=dev)
    for pad in (0, 4, 8):      # rows of 16-byte and of 8-byte alignment
        sk, sv = (torch.zeros(L, n_kv * 128 + pad, dtype=torch.bfloat16, device=dev) for _ in range(2))
        layer.decode_blocks(pool, pairs, sk, sv)
        for got, want in ((sk, k16), (sv, v16)):
            assert np.array_equal(to_u16(got[:, :n_kv * 128].contiguous()).reshape(L, n_kv, 128), want) and not to_u16(got[:, n_kv * 128:].contiguous()).any()
    layer.check()


@pytest.mark.parametrize("room", [0, -1])
@pytest.mark.parametrize("raw_groups", [256, 3])
def test_append_fills_its_window_to_the_last_byte(room, raw_groups):
    """The tile that a decode step completes needs 5 bytes a raw group: a window of exactly that many takes it, one byte less does not."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    rng = np.random.default_rng(raw_groups)
    tiers = np.zeros((1, 16, 16), int)
    tiers.reshape(-1)[rng.permutation(256)[:raw_groups]] = 3
    k16, v16 = (_tiers_to_rows(tiers, kind, rng).transpose(1, 0, 2) for kind in "kv")
    k, v = to_bf16(k16, dev), to_bf16(v16, dev)
    full = lambda b: torch.full((1, 128), b, dtype=torch.uint8)
    cache = CompressedKVCache(1, 1, 16, dict(k3=full(B3), k4=full(B4), v3=full(B3), v4=full(B4)), ovf_bytes_per_tile=5 * raw_groups + room)
    slots = torch.zeros(1, dtype=torch.int32, device=dev)
    for i in range(16): cache.append(slots, k[i:i + 1], v[i:i + 1])
    assert int(cache.overflow) == (0 if room == 0 else 2)
    for st, x16 in ((cache.k, k16), (cache.v, v16)):
        assert int(st.ovf_used[0]) == (5 * raw_groups if room == 0 else 0) and bool((st.flags != 0).any()) == (room == 0)
    if room == 0:
        dk, dv = cache.decompress(0)
        assert np.array_equal(to_u16(dk), k16) and np.array_equal(to_u16(dv), v16)


@pytest.mark.parametrize("held", [0, 1, 5, 15])
@pytest.mark.parametrize("groups", [16, 17])
def test_paged_store_completes_a_block_from_held_and_new_rows(held, groups):
    """A block of 16 or 17 four-bit groups against slots with room for 16 escape bytes, completed on top of `held` raw rows."""
    dev = require_gpu()
    from gaac_amd.paged import LayerState, build_store_entries
    rng = np.random.default_rng(held)
    tiers = np.zeros((2, 16, 16), int)
    for h in range(2): tiers[h].reshape(-1)[rng.permutation(256)[:groups]] = 1
    k16, v16 = (np.ascontiguousarray(_tiers_to_rows(tiers, kind, rng).transpose(1, 0, 2)) for kind in "kv")
    k, v = to_bf16(k16, dev), to_bf16(v16, dev)
    full = lambda b: torch.full((2, 128), b, dtype=torch.uint8)
    layer = LayerState(3, 2, 8, dict(k3=full(B3), k4=full(B4), v3=full(B3), v4=full(B4)), ovf_slot=16)
    pool = torch.full((LayerState.pool_bytes(3, 2, 16),), 255, dtype=torch.uint8, device=dev)
    entries = lambda c, n: torch.from_numpy(build_store_entries([c], [n], [[1]])).to(dev)
    if held: layer.store(k[:held], v[:held], pool, entries(0, held))
    layer.store(k[held:], v[held:], pool, entries(held, 16 - held))
    fits = groups <= 16
    assert bool((layer.mt.view(3, 4)[1] >= 0).all()) == fits and int(layer.top) == (8 if fits else 4)
    sk, sv = torch.zeros(16, 2, 128, dtype=torch.bfloat16, device=dev), torch.zeros(16, 2, 128, dtype=torch.bfloat16, device=dev)
    layer.decode_blocks(pool, torch.tensor([[1, 0, 16]], dtype=torch.int32, device=dev), sk, sv)
    assert np.array_equal(to_u16(sk), k16) and np.array_equal(to_u16(sv), v16)
    layer.check()
