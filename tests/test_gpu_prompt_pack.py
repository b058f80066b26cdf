"""Escapes of a prompt packed into the slot's windows, by the launch that adds up the tile sizes itself (up to 4096 tiles) and by the two that do it
for longer prompts, against a page of the same rows."""
import pytest
import torch

from common import to_bf16, randn_bf16
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_kv,tiles,rest", [(2, 1, 0), (2, 63, 15), (2, 64, 1), (2, 65, 0), (1, 2048, 3), (1, 2049, 0), (1, 4096, 5), (1, 4097, 5)])
def test_offsets_streams_and_counters_equal_a_page(n_kv, tiles, rest):
    dev = require_gpu()
    from gaac_amd import Codec, CompressedKVCache, TileEncoder
    L = 16 * tiles + rest
    k, v = (to_bf16(randn_bf16((L, n_kv, 128), seed=s), dev) for s in (1, 2))
    v[::97, :, ::13] *= 2.0 ** -30      # raw groups: some tiles of V have more than 64 escape bytes
    bases = {}
    for name, x in (("k", k), ("v", v)):
        c = Codec(n_kv).calibrate(x[:min(L, 512)].transpose(0, 1))
        bases[name + "3"], bases[name + "4"] = c.base3, c.base4
    cache = CompressedKVCache(2, n_kv, L + 9, bases, device=dev)
    for slot in (1, 0):
        cache.prefill(slot, k, v)
        for name, st, x in (("k", cache.k, k), ("v", cache.v, v)):
            page = TileEncoder(name).encode(Codec(n_kv).set_bases(bases[name + "3"], bases[name + "4"]), x[:16 * tiles].transpose(0, 1))
            start, h0 = page.ovf_head_start.tolist(), slot * n_kv
            assert torch.equal(st.tile_off[h0:h0 + n_kv, :tiles], page.tile_off)
            for h in range(n_kv):
                n = start[h + 1] - start[h]
                assert int(st.ovf_used[h0 + h]) == n
                at = int(st.head_start[h0 + h])
                assert torch.equal(st.ovf[at:at + n], page.ovf[start[h]:start[h] + n])
            assert torch.equal(st.tail[h0:h0 + n_kv, :rest].view(torch.int16), x[16 * tiles:].transpose(0, 1).view(torch.int16))
        assert cache.S[h0:h0 + n_kv].tolist() == [16 * tiles] * n_kv and cache.tail_len[h0:h0 + n_kv].tolist() == [rest] * n_kv
