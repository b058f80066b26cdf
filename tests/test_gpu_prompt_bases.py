"""Bases that a prompt calibrates for itself, from the tables of several blocks per head: one block and many (up to sixteen, 32, 64 and more, which are added up in
turn), none, ends of chunks, chunks at the longest length that 16-bit counts hold, every exponent there is and only one, against the histogram over all rows."""
import pytest
import torch

from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,n_kv", [(1, 1), (15, 2), (17, 3), (256, 1), (257, 1), (4099, 8), (33000, 1), (5000, 2), (700, 130), (65600, 130), (0, 1), (4096, 1), (4097, 1), (8192, 2),
                                    (8193, 1), (16383, 1), (64 * 65535 + 1, 1)])
@pytest.mark.parametrize("data", ["bits", "normal", "ones"])
def test_bases(L, n_kv, data):
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    from gaac_amd.codec import bases_from_hist, exponent_hist
    if L * n_kv > 10 ** 6 and data == "normal": pytest.skip("the other two suffice at this size")
    g = torch.Generator(device=dev).manual_seed(L + n_kv)
    def rows():
        if data == "bits": return torch.randint(-2 ** 15, 2 ** 15, (L, n_kv, 128), dtype=torch.int16, generator=g, device=dev).view(torch.bfloat16)
        if data == "ones": return torch.ones(L, n_kv, 128, dtype=torch.bfloat16, device=dev)
        scale = torch.exp2(torch.rand(1, n_kv, 128, generator=g, device=dev) * 40 - 20)
        return (torch.randn(L, n_kv, 128, generator=g, device=dev) * scale).to(torch.bfloat16)
    k, v = rows(), rows()
    cache = CompressedKVCache(2, n_kv, L + 16, ovf_bytes_per_tile=1280 if data == "bits" else 128)
    for _ in range(2): cache.prefill(1, k, v)      # the second on scratch that another prompt may have left something in
    for x, st in ((k, cache.k), (v, cache.v)):
        b3, b4 = bases_from_hist(exponent_hist(x, n_kv) if L else torch.zeros(n_kv, 128, 256, dtype=torch.int64, device=dev), n_kv)
        assert torch.equal(st.base3[n_kv:], b3) and torch.equal(st.base4[n_kv:], b4)
    if L < 10 ** 4:      # (of "bits", tiles of over a thousand escape bytes)
        for got, x in zip(cache.decompress(1), (k, v)): assert torch.equal(got.view(torch.int16), x.view(torch.int16))
