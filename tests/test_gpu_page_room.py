"""A page's escape stream against the room that it is given ahead of its size: shorter, equal, one byte longer; pages on both sides of the one-launch packing."""
import pytest
import torch

from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("H,S", [(1, 16), (3, 16 * 64 + 7), (2, 16 * 8192), (2, 16 * 8193 - 3)])
@pytest.mark.parametrize("spare", [None, 5, 0, -1, -4])      # room left; None: no escapes at all
def test_streams_around_their_room(kind, H, S, spare):
    dev = require_gpu()
    from gaac_amd import Codec, TileEncoder
    from gaac_amd.codec import STREAM_ROOM, perm, row_offsets
    n = 0 if spare is None else STREAM_ROOM * H * S - spare
    # 1.0 everywhere, with both bases at its exponent; n // 5 raw groups (five bytes) and n % 5 four-bit ones (one byte), spread over the rows
    x = torch.ones(H * S * 16, 8, dtype=torch.bfloat16, device=dev)
    at = torch.randperm(H * S * 16, generator=torch.Generator().manual_seed(S))[:n // 5 + n % 5].to(dev)
    x[at[:n // 5]] = 2.0 ** -20
    x[at[n // 5:]] = 2.0 ** 9
    # groups lie in storage order: element i of group g of a row sits in the channel that the permutation names
    rows = torch.empty(H, S, 128, dtype=torch.bfloat16, device=dev)
    rows[..., perm(kind).to(dev)] = x.view(H, S, 128)
    base = torch.full((H, 128), 127, dtype=torch.uint8, device=dev)
    page = TileEncoder(kind).encode(Codec(H).set_bases(base, base), rows)
    assert page.ovf.numel() == n + 8 and int(page.ovf_head_start[-1]) == n and not page.ovf[-8:].any()
    assert torch.equal(Codec.decode(page).view(torch.int16), rows.view(torch.int16))
    assert torch.equal(page.ovf_off, row_offsets(page.flags, S))
