"""CPU checks of the host side: the C-ABI library loads and exports every symbol the header declares, the ctypes table matches
the header's parameter lists, calls without a device fail loudly (no fallback), and the closed-form byte accounting."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gaac_hip.h")


def _declarations():
    """{name: [parameter type strings]} of every function declared in include/gaac_hip.h."""
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    out = {}
    for m in re.finditer(r"\b(?:int|const char\*)\s+(gaac_\w+)\s*\(([^;]*?)\)\s*;", text, flags=re.S):
        params = [p.strip() for p in m.group(2).replace("\n", " ").split(",")]
        out[m.group(1)] = [] if params == ["void"] else params
    return out


def test_library_exports_every_declared_symbol():
    from gaac_amd import _lib
    decl = _declarations()
    assert len(decl) >= 12 and "gaac_attn_launch" in decl and "gaac_cache_append" in decl
    assert os.path.exists(_lib.lib_path()), "build the library first: python -m gaac_amd.build"
    lib = ctypes.CDLL(_lib.lib_path())
    for name in decl:
        assert hasattr(lib, name), f"{name} is declared in include/gaac_hip.h but not exported"
    assert sorted(decl) == sorted(_lib.exported_symbols())


def test_ctypes_table_matches_the_header():
    from gaac_amd import _lib
    kind = {"int": ctypes.c_int, "long": ctypes.c_long, "float": ctypes.c_float}
    for name, params in _declarations().items():
        if name == "gaac_last_error": continue
        want = []
        for p in params:
            base = p.rsplit(" ", 1)[0].strip()
            want.append(ctypes.c_void_p if "*" in p else kind[base])
        assert _lib._SIGNATURES[name] == want, name


def test_every_entry_point_rejects_null_arguments_before_it_touches_a_device():
    """All-null, all-zero argument lists come back as -1 with a message on the calling thread: the argument checks stand in front
    of the first HIP call of every entry point.  (The two calls that only take a stream are left out: they do go to the device.)"""
    from gaac_amd import _lib
    lib = _lib.load()
    for name, args in _lib._SIGNATURES.items():
        if name in ("gaac_static_init", "gaac_static_reset"): continue
        zeros = [None if a is ctypes.c_void_p else (0.0 if a is ctypes.c_float else 0) for a in args]
        assert getattr(lib, name)(*zeros) == -1, name
        assert len(lib.gaac_last_error()) > 8, name


def test_no_device_no_fallback():
    """Without a GPU (or with CPU tensors) the product path raises instead of computing on the host."""
    from gaac_amd import Codec
    from gaac_amd.codec import exponent_hist
    x = torch.zeros(16, 2, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        exponent_hist(x, 2)
    with pytest.raises(RuntimeError):
        Codec(2, "cpu").calibrate(torch.zeros(2, 16, 128, dtype=torch.bfloat16))


@pytest.mark.parametrize("shape", [(2, 32, 64), (3, 1, 64), (2, 32, 127), (1, 1, 1), (2, 32, 256), (0, 4, 64), (4, 128), (1, 2, 32, 128)])
def test_encoder_refuses_rows_of_another_size(shape):
    """Rows that are not 128 elements are refused by every encoding call before anything is allocated for them or launched."""
    from gaac_amd import Codec, TileEncoder
    from gaac_amd.codec import encode_page, rows_in_place
    x = torch.zeros(shape, dtype=torch.bfloat16)
    base = torch.zeros(2, 128, dtype=torch.uint8)
    codec = Codec(2, "cpu").set_bases(base, base)
    if len(shape) == 3:
        with pytest.raises(RuntimeError, match="rows of 128"): encode_page(x, "k", base, base, 2)
        with pytest.raises(RuntimeError, match="rows of 128"): codec.encode(x, "v")
        with pytest.raises(RuntimeError, match="rows of 128"): TileEncoder("k", "cpu").encode(codec, x)
    with pytest.raises(RuntimeError, match="rows of 128"): TileEncoder("k", "cpu").encode_tiles(x, base, base, None, None, None, 16, 16, 2)
    with pytest.raises(RuntimeError, match="rows of 128"): rows_in_place(x, 0, 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.uint8])
def test_encoder_refuses_elements_of_another_size(dtype):
    from gaac_amd.codec import rows_in_place
    with pytest.raises(RuntimeError, match="bf16 rows"): rows_in_place(torch.zeros(2, 32, 128, dtype=dtype), 0, 1)


def test_escape_stream_beyond_32_bits_is_refused():
    """Totals are summed beyond 32 bits and refused before the stream is allocated; a head's total that reached the limit counts as too long."""
    from gaac_amd.codec import stream_bytes
    assert stream_bytes([]) == 0 and stream_bytes([5, 0, 7]) == 12 and stream_bytes([2 ** 30, 2 ** 30 - 2]) == 2 ** 31 - 2
    for totals in ([2 ** 31 - 1], [2 ** 30, 2 ** 30 - 1], [2 ** 30] * 2, [2 ** 30] * 4, [2 ** 31 - 1] * 3):
        with pytest.raises(RuntimeError, match="32-bit offsets"): stream_bytes(totals)


@pytest.mark.parametrize("H,S,off,hs,rs", [(2, 5, 0, 640, 128), (2, 5, 0, 128, 256), (3, 1, 0, 128, 7), (1, 4, 0, 3, 128), (2, 4, 8, 1024, 136), (2, 4, 0, 0, 128),
                                           (2, 4, 1, 512, 128), (2, 4, 0, 512, 129), (2, 4, 0, 513, 128), (2, 4, 0, 512, 0), (2, 4, 0, 512, 64), (2, 0, 0, 0, 128)])
def test_rows_are_read_through_strides_that_stay_inside_their_memory(H, S, off, hs, rs):
    """Every (head, row) that the returned strides address holds the 128 elements of that row, whether the rows are used where they
    are or from a copy; rows that the kernel reads are 16-byte aligned."""
    from gaac_amd.codec import rows_in_place
    mem = torch.arange(8192, dtype=torch.int16)
    x = torch.as_strided(mem, (H, S, 128), (hs, rs, 1), off)
    y, yh, yr = rows_in_place(x, 0, 1)
    assert y.data_ptr() % 16 == 0 and yh % 8 == 0 and yr % 8 == 0 and yr >= 128
    base = y.storage_offset()
    flat = torch.as_strided(y, (y.untyped_storage().nbytes() // 2,), (1,), 0)
    for h in range(H):
        for t in range(S):
            at = base + h * yh + t * yr
            assert at + 128 <= flat.numel() and torch.equal(flat[at:at + 128], x[h, t])


def test_product_code_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "gaac_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text, f"{f} mentions the test oracle"


def test_storage_index_is_a_bijection_and_perms_match_closed_forms():
    from gaac_amd.codec import storage_index, perm_k, perm_v
    for kind in ("k", "v"):
        sm, cd = storage_index(kind, "cpu")
        assert sorted(sm.tolist()) == list(range(2048)) and sorted(cd.tolist()) == list(range(768))
    pk, pv = perm_k().tolist(), perm_v().tolist()
    assert sorted(pk) == list(range(128)) and sorted(pv) == list(range(128))
    for j in range(4):
        for s in range(8):
            for q in range(4):
                assert pk[32 * j + 4 * s + q] == 16 * s + 2 * j + (0, 1, 8, 9)[q]
    for r in range(8):
        for n in range(16):
            assert pv[16 * r + n] == 8 * n + r


def test_choose_nsplit_bounds():
    from gaac_amd.kernel import choose_nsplit
    assert choose_nsplit(1, 8, 65536) == 32            # 256 blocks over 8 kv heads
    assert choose_nsplit(1, 8, 300) == 1               # never below 256 tokens per split
    assert choose_nsplit(64, 8, 65536) == 1
    assert choose_nsplit(1, 1, 1 << 20) == 256         # cap


def test_launch_nsplit_where_the_caller_leaves_the_choice():
    from gaac_amd.kernel import launch_nsplit
    for ragged in (False, True):
        assert launch_nsplit(1, 8, 65536, ragged) == 32 and launch_nsplit(4, 8, 32768, ragged) == 8      # 256 blocks
        assert launch_nsplit(1, 8, 1000, ragged) == 31 and launch_nsplit(1, 1, 8000, ragged) == 64      # 32 tokens per split, 64 splits
        for B, n_kv in ((1, 1), (32, 8), (256, 16)): assert launch_nsplit(B, n_kv, 256, ragged) == 1
        # short rows of many heads, and batches that fill the GPU without splits
        for B, n_kv, S in ((200, 2, 300), (64, 8, 2000), (48, 8, 300), (32, 8, 500), (24, 8, 1000), (65, 8, 65536), (256, 16, 4000)):
            assert launch_nsplit(B, n_kv, S, ragged) == 1, (B, n_kv, S)
        assert launch_nsplit(12, 8, 1000, ragged) == 2
    for B, n_kv, S, n in ((12, 8, 8000, 6), (24, 8, 6000, 3), (32, 8, 6000, 2), (48, 8, 2000, 2), (64, 8, 4000, 2)):
        assert launch_nsplit(B, n_kv, S, True) == n and launch_nsplit(B, n_kv, S, False) == max(1, 256 // (B * n_kv))


def test_bytes_per_slot_closed_form():
    from gaac_amd.kv_cache import CompressedKVCache
    # 8 kv heads, capacity rounded to 65552 tokens, 128 B of escape room per tile, per-sequence bases: term by term
    cap = 65552; tiles = cap // 16
    head = cap * 128 + cap * 48 + cap * 4 + tiles * 4 + tiles * 128 + 8 + 4 + 4 + 16 * 128 * 2 + 2 * 128
    assert CompressedKVCache.bytes_per_slot(8, 65537) == 8 * (2 * head + 4 + 4)
    assert CompressedKVCache.bytes_per_slot(8, 65537, per_sequence_bases=False) == 8 * (2 * (head - 256) + 8)


def test_engine_context_and_attention_layer_without_a_cache():
    """The engine-shaped surface on the host (/root/reference/nanovllm/utils/context.py:5-31): the context is one module-level object
    with the reference's fields; an attention layer without a cache refuses to run instead of falling back to anything."""
    import dataclasses
    import torch
    from gaac_amd import serving
    names = [f.name for f in dataclasses.fields(serving.Context)]
    assert names == ["is_prefill", "cu_seqlens_q", "cu_seqlens_k", "max_seqlen_q", "max_seqlen_k", "slot_mapping", "context_lens",
                     "block_tables", "kv_slots", "prefill_spans"]
    serving.set_context(True, max_seqlen_q=5, prefill_spans=[(1, 0, 5)])
    c = serving.get_context()
    assert c.is_prefill and c.max_seqlen_q == 5 and c.prefill_spans == [(1, 0, 5)] and c.kv_slots is None
    serving.reset_context()
    c = serving.get_context()
    assert not c.is_prefill and c.prefill_spans is None and c.max_seqlen_k == 0
    layer = serving.Attention(8, 128, 128 ** -0.5, 2)
    assert layer.gaac is None and layer.k_cache.numel() == 0
    q = torch.zeros(1, 8, 128, dtype=torch.bfloat16); k = torch.zeros(1, 2, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no KV cache attached"):
        layer(q, k, k)
    with pytest.raises(AssertionError, match="head_dim"):
        serving.Attention(8, 64, 0.125, 2)
    # slots from a byte budget: the closed form of the cache, no device needed for the arithmetic
    from gaac_amd.kv_cache import CompressedKVCache
    per_slot = 4 * CompressedKVCache.bytes_per_slot(8, 4096)
    assert min(16, (3 * per_slot + 5) // per_slot) == 3


@pytest.mark.parametrize("L,splits", [(20000, 92), (4000, 20), (1000, 63), (300, 2)])
def test_the_row_bound_sees_a_single_split(L, splits):
    """What the launches over ragged rows are compared with: rounding weights and output to bf16 stays far inside the bound, one split left
    out, taken twice or read from its neighbour's tokens breaks it, next to a short row with much larger outputs."""
    from common import assert_rows_close
    g = torch.Generator().manual_seed(L)
    k, v, q = (torch.randn(n, 128, generator=g, dtype=torch.float64) for n in (L, L, 4))
    p = torch.softmax(q * 0.5 @ k.T * 128 ** -0.5, -1)
    short = torch.randn(4, 128, generator=g, dtype=torch.float64)
    rows = lambda out: torch.stack([short, out])
    want = rows(p @ v)
    assert_rows_close(rows((p.bfloat16().double() @ v / p.bfloat16().double().sum(-1, keepdim=True)).bfloat16().double()), want)
    n = -(-L // splits)
    for i in (0, splits // 2, (L - 1) // n):
        w = torch.ones(L, dtype=torch.float64)
        w[i * n:(i + 1) * n] = 0.0
        at = slice(i * n, min((i + 1) * n, L))
        other = (torch.arange(at.start, at.stop) + n) % L
        for wrong in (p * w, p * (2 - w)):
            with pytest.raises(AssertionError): assert_rows_close(rows(wrong @ v / wrong.sum(-1, keepdim=True)), want)
        moved = v.clone(); moved[at] = v[other]
        with pytest.raises(AssertionError): assert_rows_close(rows(p @ moved), want)
