"""The two entry points for a prompt, called as a C program calls them: gaac_cache_prefill, whose scratch and arguments are those of its first version, against
CompressedKVCache.prefill over the edges of where its tables go; gaac_prompt_store with blocks that give up their wait."""
import pytest
import torch

from gpu_util import require_gpu
from test_gpu_short_prompts import _check, _rows, _words

pytestmark = pytest.mark.gpu
GUARD = 64


@pytest.fixture(autouse=True)
def large_blocks_go_back():
    yield
    torch.cuda.empty_cache()      # (a workspace that outlives a later test would hold on to one)


# at 102 tiles a head's escapes have room for one table, at 103 for two, at 65536 tokens one table no longer counts them
@pytest.mark.parametrize("L,n_kv", [(15, 2), (16, 1), (257, 1), (1647, 1), (1648, 1), (1648, 3), (4099, 8), (700, 130), (65535, 1), (65536, 1), (66000, 140), (30000, 2)])
@pytest.mark.parametrize("calibrate", [True, False])
def test_the_first_versions_arguments(L, n_kv, calibrate):
    dev = require_gpu()
    if L * n_kv > 10 ** 6 and not calibrate: pytest.skip("nothing depends on the length without calibration")
    from gaac_amd import CompressedKVCache, _lib
    k, v = _rows(L, n_kv, L, 1e-3), _rows(L, n_kv, L + 1, 1e-3)
    bases = None if calibrate else dict.fromkeys(("k3", "v3"), torch.full((n_kv, 128), 122)) | dict.fromkeys(("k4", "v4"), torch.full((n_kv, 128), 118))
    a, b = (CompressedKVCache(2, n_kv, L + 16, bases, ovf_bytes_per_tile=1280 if L < 1000 else 160) for _ in range(2))
    a.prefill(1, k, v)
    nt = 2 * n_kv * (L // 16)
    sizes = [2 * n_kv * 256 * 64 * 8 if calibrate else 0, nt * 1280, nt * 4, 2 * n_kv * 4]      # hist, slots, bytes of the tiles and of the heads
    scratch = [torch.full((n + GUARD,), 0xA5, dtype=torch.uint8, device=dev) for n in sizes]
    host = torch.empty(2 * n_kv, dtype=torch.int32, pin_memory=True)
    for _ in range(2):
        _lib.call("gaac_cache_prefill", *_words(b, 1, k, v), *scratch, host.data_ptr(), _lib.stream)
        _lib.call("gaac_wait_words", host.data_ptr(), 2 * n_kv, _lib.stream)
    for t, n in zip(scratch, sizes): assert (t[n:] == 0xA5).all()
    h = slice(n_kv, 2 * n_kv)
    assert torch.equal(a.S, b.S) and torch.equal(a.tail_len, b.tail_len)
    for i, (x, y) in enumerate(((a.k, b.k), (a.v, b.v))):
        for f in ("sm", "codes", "flags", "tile_off", "ovf", "ovf_used", "tail", "base3", "base4"): assert torch.equal(getattr(x, f), getattr(y, f)), f
        assert host[i * n_kv:(i + 1) * n_kv].tolist() == y.ovf_used[h].tolist()


def test_blocks_that_give_up_leave_no_prompt_that_is_reported_but_not_there():
    """After a few re-reads a block gives up: now the last block of a head, now one ahead of it.  A head is either reported and all there, or empty and told so."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache, Codec, _lib
    n_kv, L = 4, 4000
    cache = CompressedKVCache(1, n_kv, L + 16, dict.fromkeys(("k3", "v3"), torch.full((n_kv, 128), 122)) | dict.fromkeys(("k4", "v4"), torch.full((n_kv, 128), 118)),
                              ovf_bytes_per_tile=400)
    nt = 2 * n_kv * (L // 16)
    slots, sizes, heads = (torch.empty(n, dtype=torch.uint8, device=dev) for n in (nt * 1280, nt * 4, 8 * n_kv))
    host = torch.empty(2 * n_kv, dtype=torch.int32, pin_memory=True)
    rows = [(_rows(L, n_kv, i, 1e-2), _rows(L, n_kv, i + 9, 1e-2)) for i in range(3)]
    pages = [[Codec(n_kv).set_bases(st.base3, st.base4).encode(x.transpose(0, 1).contiguous(), st.kind) for st, x in ((cache.k, k), (cache.v, v))] for k, v in rows]
    told = there = 0
    for i in range(80):
        k, v = rows[i % 3]
        for st in (cache.k, cache.v): st.tile_off.fill_(-1)      # (nothing of the prompt before helps)
        _lib.call("gaac_prompt_store", *_words(cache, 0, k, v), None, 0, slots, sizes, heads, cache._scan, cache._scan.stride(0), cache._scan.shape[2], (1, 2, 3, 4, 6, 8, 12, 100)[i % 8], host.data_ptr(), _lib.stream)
        torch.cuda.synchronize()
        assert heads.view(torch.int32).tolist() == host.tolist()
        for h in range(n_kv):
            failed = [host[j * n_kv + h] < 0 for j in range(2)]
            assert int(cache.S[h]) == int(cache.tail_len[h]) == 0 if any(failed) else int(cache.S[h]) == L
            told += any(failed)
            there += not any(failed)
            for j, (st, page) in enumerate(((cache.k, pages[i % 3][0]), (cache.v, pages[i % 3][1]))):
                assert bool(cache._scan[j, h].any()) != bool(failed[j])
                if any(failed): continue
                a, b = page.ovf_head_start[h:h + 2].tolist()
                assert int(host[j * n_kv + h]) == int(st.ovf_used[h]) == b - a
                assert torch.equal(st.tile_off[h, :L // 16], page.tile_off[h]) and torch.equal(st.ovf[int(st.head_start[h]):][:b - a], page.ovf[a:b])
    print(f"heads that were told to have failed {told}, stored {there}")
    assert told and there
    for k, v in rows:
        cache.prefill(0, k, v)
        _check(cache, 0, k, v)
