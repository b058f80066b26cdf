"""Exponent histogram at the edges of its rounds: rows a wave does not have, chunks of unequal length, rows of any alignment."""
import pytest
import torch

from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_kv", [1, 3])
@pytest.mark.parametrize("S", [1, 3, 4, 5, 63, 64, 65, 127, 128, 129, 255, 257, 1000, 70001])
@pytest.mark.parametrize("shift", [0, 1, 2])      # elements that the rows are off a 16-byte boundary
def test_counts(n_kv, S, shift):
    dev = require_gpu()
    from gaac_amd.codec import exponent_hist
    g = torch.Generator(device=dev).manual_seed(S)
    bits = torch.randint(-2 ** 15, 2 ** 15, (S * n_kv * 128 + shift,), generator=g, device=dev, dtype=torch.int32).to(torch.int16)
    bits[::3] = 0x3F80      # many alike
    x = bits.view(torch.bfloat16)[shift:].view(S, n_kv, 128)
    e = (x.view(torch.int16).to(torch.int64) >> 7) & 0xFF
    want = torch.zeros(n_kv * 128, 256, dtype=torch.int64, device=dev)
    want.view(-1).index_add_(0, (torch.arange(n_kv * 128, device=dev) * 256 + e.view(S, -1)).view(-1), torch.ones(e.numel(), dtype=torch.int64, device=dev))
    assert torch.equal(exponent_hist(x, n_kv), want)


@pytest.mark.parametrize("L", [16, 65, 127, 259, 4097])
def test_bases_of_a_prompt(L):
    """The packed counts, of both kinds at once, through any strides."""
    dev = require_gpu()
    from gaac_amd import CompressedKVCache
    from gaac_amd.codec import exponent_hist, bases_from_hist
    g = torch.Generator(device=dev).manual_seed(L)
    k, v = ((torch.randn(L, 6, 128, generator=g, device=dev) * torch.exp2(torch.randint(-9, 9, (6, 128), generator=g, device=dev).float())).to(torch.bfloat16)[:, ::2] for _ in range(2))
    cache = CompressedKVCache(2, 3, L, device=dev)
    cache.prefill(1, k, v)
    for st, x in ((cache.k, k), (cache.v, v)):
        b3, b4 = bases_from_hist(exponent_hist(x, 3), 3)
        assert torch.equal(st.base3[3:], b3) and torch.equal(st.base4[3:], b4)
