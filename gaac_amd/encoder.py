"""Tile encoder on MI355X: one wave64 per (head, 16-token tile).  Public surface of /root/reference/gaac/encoder.py:79-123.

Tiers, tag words and 3-bit codes are computed in registers, sign/mantissa and code bytes are written in the native tile
order, and each tile's escape bytes go to a bounded per-tile slot (1280 B worst case); compact() packs the slots into
each head's escape stream."""
from __future__ import annotations
import torch
from . import _lib
from .codec import Codec, Page, TILE_MAX_ESC, T, rows_in_place, encode_page, perm, storage_index

SLOT = TILE_MAX_ESC


class TileEncoder:
    def __init__(self, kind: str, device="cuda"):
        self.kind = kind
        self.device = device
        self._slots = None
        self._tables = None

    def _layout(self):
        if self._tables is None:
            p = perm(self.kind).to(self.device).to(torch.int32)
            si, ci = storage_index(self.kind, self.device)
            inv_s = torch.empty_like(si); inv_s[si] = torch.arange(si.numel(), device=self.device)
            inv_c = torch.empty_like(ci); inv_c[ci] = torch.arange(ci.numel(), device=self.device)
            self._tables = (p, inv_s.to(torch.int32).contiguous(), inv_c.to(torch.int32).contiguous())
        return self._tables

    # layout tables of the reference object (the kernels do not read them: the order is compiled in)
    perm = property(lambda self: self._layout()[0])
    inv_sm = property(lambda self: self._layout()[1])
    inv_cd = property(lambda self: self._layout()[2])

    def _scratch(self, n: int, dev):
        if self._slots is None or self._slots.numel() < n:
            self._slots = torch.empty(n, dtype=torch.uint8, device=dev)
        return self._slots

    def encode_tiles(self, x, base3, base4, sm, cd, flags, S, S_pad, n_kv, bidx=None) -> torch.Tensor:
        """Encode x [H, S_in, D] (any head / token strides, e.g. a transposed view of a token-major prompt; tiles 0..ceil(S/16)-1) into sm/cd/flags with token stride S_pad; escape bytes stay in the
        scratch slots.  Returns tile_bytes int32 [H, ntiles]; finish with compact()."""
        H = x.shape[0]; ntiles = (S + T - 1) // T; dev = x.device
        x, hs, rs = rows_in_place(x, 0, 1)
        slots = self._scratch(H * ntiles * SLOT, dev)
        tile_bytes = torch.empty(H, ntiles, dtype=torch.int32, device=dev)
        _lib.call("gaac_encode_tiles", 0 if self.kind == "k" else 1, x, hs, rs, H, S, S_pad, base3, base4,
                  n_kv, bidx, sm, cd, flags, slots, tile_bytes, _lib.stream)
        return tile_bytes

    def compact(self, tile_bytes, head_start, ovf) -> torch.Tensor:
        """Pack the scratch slots into ovf at head_start[h] + tile_off[h, t]; returns tile_off int32 [H, ntiles]."""
        H, ntiles = tile_bytes.shape
        tile_off = torch.empty_like(tile_bytes)
        _lib.call("gaac_compact", self._slots, tile_bytes, tile_off, head_start, ovf,
                  H, ntiles, _lib.stream)
        return tile_off

    def encode(self, codec: Codec, x: torch.Tensor) -> Page:
        """x: [H, S, D] bf16 -> Page."""
        return encode_page(x, self.kind, codec.base3, codec.base4, codec.n_kv)
