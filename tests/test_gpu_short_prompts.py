"""Prompts whose blocks place their escapes among themselves, at the edges of the blocks (four tiles, 64 blocks) and on both sides of the lines to the two
launches (256 tiles a head, 3072 of all): every field of the slot against a page of the same rows, slots put in again and again, windows that are too small, the
epoch's wrap-around, prompts into two slots on two streams at once, replays of a graph, a wait that failed, a block that gave up."""
import pytest
import torch

from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


def _rows(L, n_kv, seed, outliers):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(L, n_kv, 128, generator=g, device="cuda")
    return torch.where(torch.rand(L, n_kv, 128, generator=g, device="cuda") < outliers, x * 1e4, x).to(torch.bfloat16)      # 0.3: a thousand escape bytes a tile


def _check(cache, slot, k, v):
    """The slot's tiles, offsets, escapes, tail and counters are those of pages of the same rows."""
    from gaac_amd import Codec
    n_kv, full = cache.n_kv, k.shape[0] // 16 * 16
    h = slice(slot * n_kv, (slot + 1) * n_kv)
    assert cache.S[h].tolist() == [full] * n_kv and cache.tail_len[h].tolist() == [k.shape[0] - full] * n_kv
    for st, x in ((cache.k, k), (cache.v, v)):
        b = h if cache.per_sequence_bases else slice(0, n_kv)
        assert torch.equal(st.tail[h, :x.shape[0] - full], x[full:].transpose(0, 1))
        if not full: continue
        page = Codec(n_kv).set_bases(st.base3[b], st.base4[b]).encode(x[:full].transpose(0, 1).contiguous(), st.kind)
        assert torch.equal(st.sm[h, :full * 128], page.sm) and torch.equal(st.codes[h, :full * 48], page.codes)
        assert torch.equal(st.flags[h, :full], page.flags) and torch.equal(st.tile_off[h, :full // 16], page.tile_off)
        start = page.ovf_head_start.tolist()
        assert st.ovf_used[h].tolist() == [b - a for a, b in zip(start, start[1:])]
        for i in range(n_kv):
            at = int(st.head_start[slot * n_kv + i])
            assert torch.equal(st.ovf[at:at + start[i + 1] - start[i]], page.ovf[start[i]:start[i + 1]])


@pytest.mark.parametrize("L,n_kv", [(16, 1), (31, 3), (63, 2), (64, 2), (65, 2), (80, 1), (1029, 2), (4096, 1), (4111, 2), (4112, 1), (1536, 16), (1552, 16), (100, 48)])
@pytest.mark.parametrize("outliers", [1e-3, 0.3])
def test_slots(L, n_kv, outliers):
    require_gpu()
    from gaac_amd import CompressedKVCache
    cache = CompressedKVCache(3, n_kv, L + 16, None if n_kv != 2 else dict.fromkeys(("k3", "v3"), torch.full((2, 128), 122)) | dict.fromkeys(("k4", "v4"), torch.full((2, 128), 118)),
                              ovf_bytes_per_tile=1280 if outliers > 0.1 else 160)
    last = {}
    for i, slot in enumerate((2, 0, 2, 2, 1)):      # (the third and fourth with fewer blocks than the launch before, and more)
        n = max(L // 2, 16) if i == 2 else L
        k, v = _rows(n, n_kv, 10 * i + L, outliers), _rows(n, n_kv, 10 * i + L + 1, outliers)
        cache.prefill(slot, k, v)
        last[slot] = k, v
    for slot, (k, v) in last.items(): _check(cache, slot, k, v)
    cache._scan[:, :, 0] = 0xFFFFFFFE      # the next epochs: 2^32 - 1, 1, 2
    for i in range(3):
        k, v = _rows(L, n_kv, 99 + i, outliers), _rows(L, n_kv, 199 + i, outliers)
        cache.prefill(0, k, v)
        _check(cache, 0, k, v)
    assert cache._scan[:, :n_kv, 0].unique().numel() == 1


@pytest.mark.parametrize("many", ["k", "v", "both"])
def test_windows_that_have_to_grow(many):
    require_gpu()
    from gaac_amd import CompressedKVCache
    cache = CompressedKVCache(2, 2, 640, ovf_bytes_per_tile=40)
    k0, v0 = _rows(333, 2, 1, 1e-3), _rows(333, 2, 2, 1e-3)
    cache.prefill(1, k0, v0)
    cap = cache.k.ovf_cap
    k, v = _rows(600, 2, 3, 0.3 if many != "v" else 1e-3), _rows(600, 2, 4, 0.3 if many != "k" else 1e-3)
    cache.prefill(0, k, v)
    assert cache.k.ovf_cap == cache.v.ovf_cap > cap
    _check(cache, 0, k, v)
    _check(cache, 1, k0, v0)


def _words(cache, slot, k, v):
    """The arguments that gaac_prompt_store and gaac_cache_prefill both take, up to the stores'."""
    L, n_kv = k.shape[0], cache.n_kv
    return [k, v, 128, n_kv * 128, 128, n_kv * 128, L, n_kv, slot * n_kv, cache.cap, cache.k.ovf_cap, cache.k.base3.shape[0], int(cache.per_sequence_bases), cache.tail_len, cache.S,
            cache.k.head_start, *cache.k.kernel_args(), *cache.v.kernel_args()]


def _bases(n_kv): return dict.fromkeys(("k3", "v3"), torch.full((n_kv, 128), 122)) | dict.fromkeys(("k4", "v4"), torch.full((n_kv, 128), 118))


def _scratch(L, n_kv):
    """Slots, bytes of the tiles, bytes of the heads."""
    nt = 2 * n_kv * (L // 16)
    return [torch.empty(n, dtype=torch.uint8, device="cuda") for n in (nt * 1280, nt * 4, 8 * n_kv)]


def test_two_streams():
    require_gpu()
    from gaac_amd import CompressedKVCache
    cache = CompressedKVCache(2, 8, 800)
    rows = [[_rows(777, 8, 10 * i + j, 1e-3) for j in range(2)] for i in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(20):
        for slot, s in enumerate(streams):
            with torch.cuda.stream(s): cache.prefill(slot, *rows[slot])
    torch.cuda.synchronize()
    for slot in range(2): _check(cache, slot, *rows[slot])


def test_two_streams_at_once():
    """Launches of two slots in flight together: both streams wait for a third before each pair, and the host waits for neither until both have theirs."""
    require_gpu()
    from gaac_amd import CompressedKVCache, _lib
    cache = CompressedKVCache(2, 8, 800, _bases(8))
    rows = [[[_rows(777, 8, 10 * i + j, 1e-3) for j in range(2)] for i in range(2)] for _ in range(3)]
    streams, first = [torch.cuda.Stream() for _ in range(2)], torch.cuda.Stream()
    scratch, host = [_scratch(777, 8) for _ in range(2)], [torch.empty(16, dtype=torch.int32, pin_memory=True) for _ in range(2)]
    torch.cuda.synchronize()
    for n in range(30):
        with torch.cuda.stream(first): torch.cuda._sleep(5000000)
        for s in streams: s.wait_stream(first)
        for slot in ((0, 1), (1, 0))[n % 2]:
            _lib.call("gaac_prompt_store", *_words(cache, slot, *rows[n % 3][slot]), None, 0, *scratch[slot], cache._scan[0, 8 * slot:], cache._scan.stride(0), cache._scan.shape[2], 0,
                      host[slot].data_ptr(), streams[slot].cuda_stream)
        assert n == 0 or all((h < 0).any() for h in host)      # (neither is through; the first pair sets the streams up)
        for slot in range(2): _lib.call("gaac_wait_words", host[slot].data_ptr(), 16, streams[slot].cuda_stream)
        for slot in range(2): _check(cache, slot, *rows[n % 3][slot])


def test_replays_of_a_graph():
    """The launches of a prompt in a graph (without words on the host, which nothing in it could wait for), replayed over new rows, with prompts outside it between the replays."""
    require_gpu()
    from gaac_amd import CompressedKVCache, _lib
    cache = CompressedKVCache(2, 3, 800, _bases(3))
    k, v, scratch = _rows(777, 3, 1, 1e-3), _rows(777, 3, 2, 1e-3), _scratch(777, 3)
    def store(stream):
        _lib.call("gaac_prompt_store", *_words(cache, 1, k, v), None, 0, *scratch, cache._scan[0, 3:], cache._scan.stride(0), cache._scan.shape[2], 0, None, stream)
    store(_lib.stream)
    _check(cache, 1, k, v)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph): store(_lib.stream)
    for n in range(5):
        other = _rows(100 + 150 * n, 3, 50 + n, 1e-3), _rows(100 + 150 * n, 3, 60 + n, 1e-3)
        cache.prefill(n % 2, *other)      # into the graph's slot, into the other
        if n % 2 == 0: _check(cache, 0, *other)
        k.copy_(_rows(777, 3, 10 + n, 1e-3))
        v.copy_(_rows(777, 3, 20 + n, 1e-3))
        graph.replay()
        if n == 3: graph.replay()
        torch.cuda.synchronize()
        _check(cache, 1, k, v)


@pytest.mark.parametrize("through", ["binding", "python"])
def test_a_failed_wait_leaves_the_slot_armed(through, monkeypatch):
    require_gpu()
    from gaac_amd import CompressedKVCache, _lib
    cache = CompressedKVCache(3, 2, 320)
    k, v = _rows(300, 2, 1, 1e-3), _rows(300, 2, 2, 1e-3)
    for slot in range(3): cache.prefill(slot, k, v)
    armed = cache._scan.clone()
    binding, call = _lib.calls(), _lib.call
    class Calls:
        def __getattr__(self, name): return getattr(binding, name)
        def prompt_store(self, *a):
            if through == "python": return None
            binding.prompt_store(*a)
            raise RuntimeError("gaac_wait_words failed")
    def fail(name, *a):
        call(name, *a)
        if name == "gaac_wait_words": raise RuntimeError("gaac_wait_words failed")
    with monkeypatch.context() as m:
        m.setattr(_lib, "_calls", Calls())
        m.setattr(_lib, "call", fail)
        with pytest.raises(RuntimeError, match="gaac_wait_words"): cache.prefill(1, k, v)
    assert not cache._scan[:, 2:4].any() and torch.equal(cache._scan[:, :2], armed[:, :2]) and torch.equal(cache._scan[:, 4:], armed[:, 4:])
    cache.prefill(1, v, k)
    _check(cache, 1, v, k)


@pytest.mark.parametrize("through", ["binding", "python"])
@pytest.mark.parametrize("kind", [0, 1])
def test_a_block_that_gave_up_fails_the_prompt_wherever_it_stands(kind, through, monkeypatch):
    """The mark of a block that gave up, left by the host: the launch itself finds all words, as the last block does if it looks late enough."""
    require_gpu()
    from gaac_amd import CompressedKVCache, _lib
    cache = CompressedKVCache(2, 3, 600)
    k, v = _rows(577, 3, 1, 1e-3), _rows(577, 3, 2, 1e-3)      # nine blocks a head and a tail
    for slot in range(2): cache.prefill(slot, k, v)
    cache._scan[kind, 4, 0] += 1 << 32      # slot 1, head 1
    other = cache._scan[:, :3].clone()
    with monkeypatch.context() as m:
        if through == "python": m.setattr(_lib, "_calls", _lib._CtypesCalls())
        m.setattr(cache, "_rearm", lambda slot: None)      # the device has it done
        with pytest.raises(RuntimeError, match="gaac_wait_words"): cache.prefill(1, v, k)
    assert cache.S.tolist() == [576] * 4 + [0, 576] and cache.tail_len.tolist() == [1] * 4 + [0, 1]
    assert not cache._scan[kind, 4].any() and torch.equal(cache._scan[:, :3], other) and cache._scan[1 - kind, 4].any()
    for n in (577, 100, 577):
        cache.prefill(1, v[:n], k[:n])
        _check(cache, 1, v[:n], k[:n])
    _check(cache, 0, k, v)
