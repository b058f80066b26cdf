"""Encoder and escape packing at the sizes where their launches change shape: rows through the caches or past them (8192 tiles), the packing's
blocks of 64 tiles and waves of 16, the scan's rounds of 4096 tiles, tiles with more than 64 escape bytes, ragged last tiles."""
import numpy as np
import pytest
import torch

from oracle import gaac_oracle as O
from common import kv_like16, to_bf16, to_u16
from gpu_util import require_gpu, native_to_reference_page, assert_pages_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("S", [1, 16, 17, 16 * 15 + 3, 16 * 63, 16 * 64 + 1, 16 * 130])
@pytest.mark.parametrize("outliers", [1e-3, 0.3])
def test_pages_at_the_packing_edges_equal_the_oracle(kind, S, outliers):
    dev = require_gpu()
    from gaac_amd import Codec, TileEncoder
    n_kv = 3
    x16 = kv_like16(n_kv, S, seed=S, outliers=outliers)      # 0.3: most groups are raw, 1000 escape bytes a tile
    codec = Codec(n_kv).calibrate(to_bf16(kv_like16(n_kv, 512, seed=5)))
    page = TileEncoder(kind).encode(codec, to_bf16(x16, dev))
    want = O.encode(x16, kind, codec.base3.cpu().numpy(), codec.base4.cpu().numpy(), n_kv)
    assert_pages_equal(native_to_reference_page(page), want)
    assert not page.ovf[-8:].any()
    assert np.array_equal(to_u16(Codec.decode(page)), x16)


@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("H,S", [(1, 16 * 4096 + 5), (2, 16 * 4095), (5, 16 * 1700 - 1)])
def test_many_tiles(kind, H, S):
    """More tiles than one round of the scan, and launches on both sides of the encoder's switch: the tables follow from the tag words,
    the rows come back."""
    dev = require_gpu()
    from gaac_amd import Codec, TileEncoder
    from gaac_amd.codec import row_offsets
    g = torch.Generator(device=dev).manual_seed(S)
    x = (torch.randn(H, S, 128, generator=g, device=dev) * torch.exp2(torch.rand(H, 1, 128, generator=g, device=dev) * 8 - 4)).to(torch.bfloat16)
    page = TileEncoder(kind).encode(Codec(H).calibrate(x[:, :1024]), x)
    assert torch.equal(Codec.decode(page).view(torch.int16), x.view(torch.int16))
    assert torch.equal(page.ovf_off, row_offsets(page.flags, S))
    rows = row_offsets(page.flags, page.flags.shape[1])
    assert torch.equal(page.tile_off, rows[:, ::16])
    f = page.flags[:, -1].to(torch.int64)
    last = sum((((f >> (2 * j)) & 1) + 4 * ((f >> (2 * j + 1)) & 1)) for j in range(16))
    start = torch.cat([torch.zeros(1, dtype=torch.int64, device=dev), (rows[:, -1] + last).cumsum(0)])
    assert torch.equal(page.ovf_head_start.to(torch.int64), start) and page.ovf.numel() == int(start[-1]) + 8


@pytest.mark.parametrize("ntiles", [4096, 3 * 4096 - 7])
def test_scan_totals_stop_at_the_largest_int(ntiles):
    """Totals that 32 bits cannot hold come out as 2^31 - 1, next to heads whose totals are exact up to there."""
    dev = require_gpu()
    from gaac_amd import _lib
    big = (2 ** 31 - 2) // ntiles
    per_tile = [3, big, min(big + 1 + big // 8, 2 ** 18), 2 ** 18]      # per head; a round of 4096 tiles stays below 2^31
    sizes = torch.tensor(per_tile, dtype=torch.int32, device=dev)[:, None].expand(4, ntiles).contiguous()
    sizes[1] = min(big, 2 ** 18)
    off, heads, host = torch.empty_like(sizes), torch.empty(4, dtype=torch.int32, device=dev), torch.empty(4, dtype=torch.int32, pin_memory=True)
    _lib.call("gaac_tile_scan", _lib.ptr(sizes), 4, ntiles, _lib.ptr(off), _lib.ptr(heads), host.data_ptr(), _lib.stream())
    torch.cuda.synchronize()
    exact = sizes.cpu().to(torch.int64)
    want = exact.sum(1).clamp(max=2 ** 31 - 1)
    assert heads.tolist() == host.tolist() == want.tolist()
    assert ntiles == 4096 or (want[2:] == 2 ** 31 - 1).all()
    for h in range(4):
        if want[h] < 2 ** 31 - 1: assert torch.equal(off[h].cpu().to(torch.int64), exact[h].cumsum(0) - exact[h])
