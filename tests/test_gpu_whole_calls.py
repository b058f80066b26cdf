"""Calls that the binding makes as a whole against the same calls through Python (ctypes), over the forms that either takes: contiguous tensors, strided and
misaligned ones, other shapes of the slot map, escape streams beyond the room, and what is refused.  Which calls the binding makes, and which it gives back, is checked as well."""
import warnings

import pytest
import torch

from gaac_amd import _lib
from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


WHOLE = ("attend", "token_append", "prompt_store", "page_encode", "page_decode")


@pytest.fixture
def both(monkeypatch):
    """both(f): f's results with the binding and with Python's calls; both.made: for each whole call that f came to, whether the binding made it."""
    binding = _lib.calls()
    assert hasattr(binding, "bind")
    class Watched:
        def __getattr__(self, name):
            def call(*a):
                out = getattr(binding, name)(*a)
                if name in WHOLE: run.made.setdefault(name, []).append(out is not None)
                return out
            return call
    def run(f):
        out, run.made = [], {}
        for calls in (Watched(), _lib._CtypesCalls()):
            monkeypatch.setattr(_lib, "_calls", calls)
            try: out.append(f())
            except (RuntimeError, AssertionError, TypeError) as e: out.append((type(e), str(e)))
        monkeypatch.setattr(_lib, "_calls", binding)
        return out
    return run


def _rows(shape, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(torch.bfloat16)


def _same(a, b):
    assert type(a) is type(b)
    if isinstance(a, torch.Tensor): assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a.view(torch.int16) if a.dtype == torch.bfloat16 else a, b.view(torch.int16) if b.dtype == torch.bfloat16 else b)
    elif isinstance(a, (tuple, list)):
        assert len(a) == len(b)
        for x, y in zip(a, b): _same(x, y)
    else: assert a == b


FORMS = {      # of rows [n, heads, 128]
    "plain": lambda n, h, seed: _rows((n, h, 128), seed),
    "token stride": lambda n, h, seed: _rows((n, h + 1, 128), seed)[:, :h],
    "head-major": lambda n, h, seed: _rows((h, n, 128), seed).transpose(0, 1),
    "misaligned": lambda n, h, seed: _rows((n * h * 128 + 1,), seed)[1:].view(n, h, 128),
    "reversed channels": lambda n, h, seed: _rows((n, 128, h), seed).transpose(1, 2),
    "float": lambda n, h, seed: _rows((n, h, 128), seed).float(),
}
IN_PLACE = ("plain", "token stride", "head-major")      # what the encoder reads where it lies
CONTIGUOUS = ("plain", "misaligned")


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("kind", ["k", "v"])
def test_pages(both, form, kind):
    require_gpu()
    from gaac_amd import Codec, TileEncoder, attention
    x = FORMS[form](333, 2, 1).transpose(0, 1)
    other = _rows((2, 333, 128), 2)
    codec = Codec(2).calibrate(other)
    q = FORMS[form](2, 8, 3)[:1]
    def f():
        p = TileEncoder(kind).encode(codec, x)
        w = TileEncoder("v" if kind == "k" else "k").encode(codec, other)
        out = attention(q, *((p, w) if kind == "k" else (w, p)))
        return [getattr(p, n) for n in ("sm", "codes", "flags", "ovf_off", "ovf", "ovf_head_start", "tile_off", "H", "S", "n_kv", "kind")], Codec.decode(p), out
    a, b = both(f)
    _same(a, b)
    if form == "float": assert a[0] is RuntimeError and both.made == dict(page_encode=[False])
    else: assert both.made == dict(page_encode=[form in IN_PLACE, True], attend=[form in CONTIGUOUS or form == "token stride"], page_decode=[True])      # (the query is a single row)


def test_a_stream_beyond_its_room(both):
    require_gpu()
    from gaac_amd import Codec
    x = torch.randint(-2 ** 15, 2 ** 15, (2, 100, 128), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).to(torch.int16).view(torch.bfloat16)
    codec = Codec(1).set_bases(torch.zeros(1, 128), torch.full((1, 128), 17))
    def f():
        p = codec.encode(x, "k")
        assert p.ovf.numel() > 3 * 200 + 8
        return p.ovf[:-8], p.tile_off, Codec.decode(p).view(torch.int16)
    a, b = both(f)
    _same(a, b)
    assert torch.equal(a[2], x.view(torch.int16)) and both.made == dict(page_encode=[True], page_decode=[True])


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("L", [15, 16, 333])
@pytest.mark.parametrize("calibrate", [False, True])
def test_cache(both, form, L, calibrate):
    require_gpu()
    from gaac_amd import CompressedKVCache, Codec
    c = Codec(2).calibrate(_rows((2, 500, 128), 9))
    bases = None if calibrate else dict(k3=c.base3, k4=c.base4, v3=c.base3, v4=c.base4)
    k, v, q = FORMS[form](L, 2, 1), FORMS[form](L, 2, 2), FORMS[form](2, 8, 3)
    new = FORMS[form](2, 2, 4)
    def f(slots):
        def run():
            cache = CompressedKVCache(3, 2, 400, bases, ovf_bytes_per_tile=16)      # (333 tokens: windows that have to grow)
            cache.prefill(2, k, v)
            cache.prefill(0, k, v)
            for _ in range(3): cache.append(slots, new, new)
            out = cache.attention(q, slots, 128 ** -0.5)
            cache.check_capacity()
            return [out, cache.k.ovf_cap, cache.S, cache.tail_len, *cache.decompress(0), *cache.decompress(2)]
        return run
    i = dict(dtype=torch.int32, device="cuda")
    for slots in (torch.tensor([2, 0], **i), torch.tensor([[2], [-1]], **i), torch.tensor([2, 9, 0, 9], **i)[::2].contiguous(), torch.tensor([2], **i)):
        a, b = both(f(slots))
        _same(a, b)
        made = both.made
        if form == "float" and L >= 16:
            assert a[0] is RuntimeError and not made      # refused ahead of the call
            continue
        assert made["prompt_store"] == [L >= 16 and form in IN_PLACE] * 2
        if slots.numel() == 1 or form == "float":
            assert a[0] is RuntimeError and made["token_append"] == [False] and len(made) == 2
            continue
        assert made["token_append"] == [form in CONTIGUOUS] * 3 and made["attend"] == [form in CONTIGUOUS and slots.dim() == 1]
        assert all(made.get("page_decode", [True])) and (L < 16 or len(made["page_decode"]) == 4)


def test_tensors_without_an_address_and_a_lack_of_memory_raise_as_through_python(both):
    require_gpu()
    from gaac_amd import Codec, CompressedKVCache, attention
    x = _rows((2, 200000, 128), 1)
    torch.cuda.empty_cache()      # (no large segment that is only partly in use)
    codec = Codec(2).calibrate(x)
    K, V = codec.encode(x, "k"), codec.encode(x, "v")
    cache, slots = CompressedKVCache(2, 2, 64, dict(k3=codec.base3, k4=codec.base4, v3=codec.base3, v4=codec.base4)), torch.tensor([1], dtype=torch.int32, device="cuda")
    q, new = _rows((3, 1, 8, 128), 2), _rows((3, 1, 2, 128), 3)
    def refused(f):
        try: f()
        except Exception as e: return type(e)
    def vmaps():
        return [refused(lambda: torch.vmap(lambda t: attention(t, K, V))(q)), refused(lambda: torch.vmap(lambda t: cache.append(slots, t, t))(new)), cache.S.tolist(), cache.tail_len.tolist()]
    a, b = both(vmaps)
    assert a == b and a[0] is not None and a[1] is not None
    def no_room():
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 4096) / torch.cuda.get_device_properties(0).total_memory)
        try: return refused(lambda: Codec.decode(K)), refused(lambda: codec.encode(x, "k"))
        finally: torch.cuda.set_per_process_memory_fraction(1.0)
    assert both(no_room) == [(torch.OutOfMemoryError,) * 2] * 2
