"""The page encoder at the edges of its blocks (four tiles, one a wave) and on both sides of the line from which rows are read past the caches, with bases
over their whole range: differences of exponents reach from -255 to 255."""
import numpy as np
import pytest
import torch

from oracle import gaac_oracle as O
from common import to_bf16, to_u16
from gpu_util import require_gpu, native_to_reference_page, assert_pages_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("H,S", [(1, 1), (2, 16), (1, 17), (3, 63), (2, 64), (1, 65), (2, 79), (2, 81), (16, 8191), (15, 8190)])      # 8192 tiles; 7680
def test_encode(kind, H, S):
    dev = require_gpu()
    from gaac_amd import Codec
    rng = np.random.default_rng(100 * H + S)
    n_kv = 1 if H == 15 else H
    b3, b4 = (rng.integers(0, 256, (n_kv, 128), dtype=np.uint8) for _ in range(2))
    b3[:, ::7], b4[:, ::5], b3[:, 3::9], b4[:, 3::9] = 255, 0, 0, 255
    base = np.where(rng.random((H, S, 16, 1)) < 0.5, 0, 1)      # per group of adjacent channels: exponents at the 3-bit bases, or at the 4-bit ones
    near = np.where(np.repeat(base, 8, -1).reshape(H, S, 128) == 0, np.tile(b3, (H // n_kv, 1))[:, None], np.tile(b4, (H // n_kv, 1))[:, None]).astype(np.int64)
    e = (near + rng.integers(0, 8, (H, S, 128)) + 8 * (rng.random((H, S, 128)) < 0.01)) % 256
    e = np.where(rng.random((H, S, 128)) < 0.002, rng.integers(0, 256, (H, S, 128)), e)
    x16 = (rng.integers(0, 2, (H, S, 128)) << 15 | e << 7 | rng.integers(0, 128, (H, S, 128))).astype(np.uint16)
    codec = Codec(n_kv, dev).set_bases(torch.from_numpy(b3), torch.from_numpy(b4))
    page = codec.encode(to_bf16(x16, dev), kind)
    assert np.array_equal(to_u16(Codec.decode(page)), x16)
    if H * S < 1000: assert_pages_equal(native_to_reference_page(page), O.encode(x16, kind, b3, b4, n_kv))
    else:      # (the reordering of a page is slow in Python: the sizes of the tiles only)
        want = O.encode(x16, kind, b3, b4, n_kv)
        assert np.array_equal(page.tile_off.cpu().numpy(), want.tile_off) and np.array_equal(page.ovf_head_start.cpu().numpy(), want.ovf_head_start)
