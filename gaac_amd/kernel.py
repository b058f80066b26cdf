"""Fused decode attention over the compressed KV on MI355X.  Public surface of /root/reference/gaac/kernel.py:332-359.

attention() launches the split-K kernel (one block per (batch row, kv head, split), MFMA score and output products on
K/V decoded in registers, optional raw-BF16 tail as one more block row; the last block of a kv head to finish merges
the partials) on the current stream, with no host synchronization.  Cache heads are addressed through a slot map exactly as in the reference: batch row b
reads cache head SLOT[b]*n_kv + kvh, SLOT[b] < 0 = padded row (output 0)."""
from __future__ import annotations
import functools
import torch
from . import _lib

D = 128
GMAX = 16
MAX_SPLITS = 1024


class _Ext:
    """What the reference's `_ext()` returns (/root/reference/gaac/kernel.py:332-337): an object whose
    `gaac_attn_launch(<16 store tensors>, q, slot, n_q, n_kv, SL, S_pad, scale, nsplit, kt, vt, TL, TCAP) -> Tensor` has the tensor
    signature and behaviour of the reference's pybind entry (kernel.py:296-326): it checks the GQA group and the head dim, allocates the
    output ([B*n_q, 128], dtype of q), takes the raw tail when `kt.numel() > 0`, launches on the current stream without synchronizing
    and returns the output.  The calls of /root/reference/gaac/kernel.py:355 and kv_cache.py:188 work on it unchanged.
    `lib` is the loaded C library (ctypes.CDLL) for callers that want the raw entry points."""
    def __init__(self, lib):
        self.lib = lib

    def gaac_attn_launch(self, smk, ck, fk, tok, ovk, ohsk, b3k, b4k, smv, cv, fv, tov, ovv, ohsv, b3v, b4v,
                         q, slot, n_q, n_kv, SL, S_pad, scale, nsplit, kt, vt, TL, TCAP):
        G = n_q // max(1, n_kv)
        if not (1 <= G <= GMAX and G * n_kv == n_q):
            raise RuntimeError(f"GQA group size must be 1..{GMAX}")
        if q.shape[-1] != D:
            raise RuntimeError("head_dim must be 128")
        B = slot.shape[0]
        has_tail = kt.numel() > 0
        out = torch.empty(B * n_q, D, dtype=q.dtype, device=q.device)
        ws = shared_workspace(B * n_q, nsplit, q.dtype, q.device)
        _lib.call("gaac_attn_fused", smk, ck, fk, tok, ovk, ohsk, b3k, b4k, smv, cv, fv, tov, ovv, ohsv, b3v, b4v,
                  q, slot, B, n_q, n_kv, SL, int(S_pad), float(scale), int(nsplit), b3k.shape[0],
                  kt if has_tail else None, vt if has_tail else None, TL if has_tail else None, int(TCAP) if has_tail else 0,
                  -1, ws.pm, ws.pl, ws.pa, ws.epoch, out, _lib.stream)
        return out


_ext_obj = None


def _ext():
    """The native extension in the shape of the reference's (raises if the library is not built)."""
    global _ext_obj
    if _ext_obj is None: _ext_obj = _Ext(_lib.load())
    return _ext_obj


def choose_nsplit(B: int, n_kv: int, S: int, target_ctas: int = 256, min_tok: int = 256, cap: int = 256) -> int:
    """Splits per (row, kv head): one eight-wave block per CU of the 256-CU MI355X (the reference targets 96 CTAs for a 48-SM
    part, kernel.py:340-342), at least min_tok tokens per split.  Launches of up to 256 blocks use eight-wave blocks, larger
    ones four-wave blocks (two per CU)."""
    return min(max(1, target_ctas // (B * n_kv)), max(1, S // min_tok), cap)


@functools.lru_cache(maxsize=1024)
def launch_nsplit(B: int, n_kv: int, S: int, ragged: bool) -> int:
    """Splits per (row, kv head) where the caller leaves the choice: S tokens per row, or up to S if ragged (the launch then shares its
    blocks out by length).  Measured, 4 query heads per kv head, us:
      * up to 256 tokens in one split (100 tokens: 6.8, against 7.3 to 8.8 with 2 to 6 splits; 300 tokens: 9.0, against 8.2 with 8);
      * at least 32 tokens per split (1000 tokens x 8 heads: 11.3 with 3 splits, 9.0 with 6, 8.7 with 32; 3000: 11.3 with 12, 9.5 with
        32), but no more than 64 splits of less than 256 (the merge: 8000 tokens, 1 head of 16 queries: 14.7 with 64, 24.4 with 256);
      * one eight-wave block per CU (256 blocks: a second round of blocks costs more than it evens out);
      * ragged rows whose heads alone take more than a quarter of the CUs: two four-wave blocks per CU, to have enough of them to share
        out, once the rows are long enough to pay for more starts and merges.  x 8 heads, one block per CU / two: 12 rows of 300..8000
        tokens 43.6 / 33.3, 24 of 300..6000 81 / 48, 24 of 300..3000 45 / 30, 32 of 300..6000 82.5 / 58, 32 of 100..2000 33.3 / 27.0;
        but 12 of 100..1000 15.3 / 15.6, 16 of 1000 16.9 / 17.3, 32 of 100..500 14.0 / 17.3.  Where long rows turn out equal it
        costs little (24 of 3000: 47.6 / 48.7, 32 of 3000: 52.3 / 52.2, 24 of 12000: 159 / 162; 28 of 4000..5000: 73.6 / 68.1);
      * ragged, more heads than CUs: two splits, one / two: 48 rows of 300..8000 x 8 heads 157 / 117, 48 of 100..2000 47.7 / 38.0, 64 of
        200..4000 86.2 / 86.4, 64 of 100..2000 50.4 / 48.6; but 200 of 300 x 2 heads 16.5 / 17.1.  Equal: 48 of 2000 59.6 / 59.1."""
    H = B * n_kv
    if S <= 256: return 1
    if ragged and B > 1 and 64 < H <= 256 and S >= max(1500, 7 * H): n = -(-512 // H)
    elif ragged and B > 1 and (256 < H <= 384 and S >= 1000 or 384 < H <= 512 and S >= 4000): n = 2
    else: n = 256 // H
    return max(1, min(n, max(S // 256, min(64, S // 32))))


class AttnWorkspace:
    """Output + split partials of one launch shape (rows = B*n_q).  The one-kernel launch stores every partial value as a 64-bit
    record (fp32 bits | launch epoch << 32): pm, pl [rows*NSLOT], pa [rows*NSLOT*D] int64.  epoch: [0] the epoch of the last merged
    one-kernel launch on this workspace, [1] failure bits that a launch sets instead of hanging (bit 0: a merging block gave up
    waiting for a partial and wrote its rows as NaN; bit 1: the epoch could not be advanced), [2 + i] the arrival mark of block i of
    the launch (rows*NSLOT words: a launch has B*n_kv*NSLOT <= rows*NSLOT blocks).  The two-kernel launch
    (phase "split" / "combine" / "both") keeps plain fp32 partials in buffers of its own, made on first use, so that its values can
    never be taken for records."""
    def __init__(self, rows: int, nslot: int, dtype, dev, with_out: bool = True):
        self.rows, self.nslot, self.dev = rows, nslot, dev
        self.out = torch.empty(rows, D, dtype=dtype, device=dev) if with_out else None      # None: a fresh output per launch
        self.pm = torch.zeros(rows * nslot, dtype=torch.int64, device=dev)
        self.pl = torch.zeros(rows * nslot, dtype=torch.int64, device=dev)
        self.pa = torch.zeros(rows * nslot * D, dtype=torch.int64, device=dev)
        self.epoch = torch.zeros(2 + rows * nslot, dtype=torch.int32, device=dev)
        self._f32 = None

    def f32_partials(self):
        """fp32 pm, pl, pa of the two-kernel launch (allocated on first use)."""
        if self._f32 is None:
            n = self.rows * self.nslot
            self._f32 = tuple(torch.empty(k, dtype=torch.float32, device=self.dev) for k in (n, n, n * D))
        return self._f32

    def failure_bits(self) -> int:
        """Host read of the failure word (synchronizes with the device)."""
        return int(self.epoch[1])

    def check(self, bits: int | None = None):
        """Raises if a one-kernel launch on this workspace gave up a wait since the last reset() (its output rows are NaN, or the
        epoch stands still); poll it where the engine polls its other device-side error words.  bits: failure_bits() if the
        caller fetched them already."""
        if bits is None: bits = self.failure_bits()
        if bits:
            raise RuntimeError("fused decode attention gave up waiting for" + (" a split's partial (rows written as NaN)" if bits & 1 else "") +
                               (" the other blocks of the launch (epoch not advanced)" if bits & 2 else "") +
                               "; the workspace may hold records of a wrong epoch: re-arm with reset()")

    def reset(self):
        """Re-arm after a failed launch: the epochs, the failure bits and the records start from zero again."""
        for t in (self.pm, self.pl, self.pa, self.epoch): t.zero_()


_SHARED_WS_MAX = 8            # launch shapes whose workspace is kept per process; the least recently used one goes first
_shared_ws: dict = {}


def shared_workspace(rows: int, nslot: int, dtype, dev) -> AttnWorkspace:
    """The workspace that callers who pass none share: one per (device, launch shape, stream), zeroed once when it is made (a fresh
    buffer per call would have to be cleared per call: recycled memory may hold records whose epoch matches a new counter), at most
    _SHARED_WS_MAX of them (least recently used first out).  It has no output buffer of its own, so every launch returns a fresh
    tensor.  A workspace is never made while the stream is capturing (its memory and its zeroing would end up inside the graph):
    callers that capture pass their own, as CompressedKVCache and LayerState do."""
    dev = torch.device(dev)
    index = dev.index if dev.index is not None else torch.cuda.current_device()
    key = (dev.type, index, rows, nslot, dtype, torch._C._cuda_getCurrentRawStream(index))
    ws = _shared_ws.pop(key, None)
    if ws is None:
        if torch.cuda.is_current_stream_capturing():
            raise RuntimeError("no attention workspace for this launch shape yet and the stream is capturing: run the launch once before "
                               "the capture, or pass a workspace (AttnWorkspace) of your own")
        ws = AttnWorkspace(rows, nslot, dtype, dev, with_out=False)
        while len(_shared_ws) >= _SHARED_WS_MAX: _shared_ws.pop(next(iter(_shared_ws)))
    _shared_ws[key] = ws      # most recently used last
    return ws


def _store_args(st):
    hs = st.head_start if hasattr(st, "head_start") else st.ovf_head_start
    return st.sm, st.codes, st.flags, st.tile_off, st.ovf, hs, st.base3, st.base4


def attn_launch(K, V, q2d, slots, n_q, n_kv, SL, S_pad, scale, nsplit, kt=None, vt=None, TL=None, TCAP=0, ws=None, phase="fused", S_all=-1, out=None):
    """K, V: objects with sm, codes, flags, tile_off, ovf, head_start|ovf_head_start, base3, base4 (a Page or a cache store).
    q2d: [B*n_q, D] or [B, n_q, D] bf16 contiguous.  Returns out, or if none is given [B*n_q, D] bf16.  phase: "fused" (one kernel, one block of each
    kv head merges) | "both" (split kernel then merge kernel) | "split" | "combine" (the halves of "both").
    S_all >= 0: every addressed head holds exactly S_all compressed tokens (SL is not read by the one-kernel launch)."""
    G = n_q // max(1, n_kv)
    if not (1 <= G <= GMAX and G * n_kv == n_q):
        raise RuntimeError(f"GQA group size must be 1..{GMAX}")
    if q2d.shape[-1] != D:
        raise RuntimeError("head_dim must be 128")
    B = slots.shape[0] if slots is not None else q2d.numel() // (n_q * D)      # slots=None: row b attends over cache heads b*n_kv ..
    has_tail = kt is not None and kt.numel() > 0
    nslot = nsplit        # the raw tail is folded into the last split's partial
    if ws is None:
        ws = shared_workspace(B * n_q, nslot, q2d.dtype, q2d.device)
    elif ws.rows != B * n_q or ws.nslot != nslot:
        raise RuntimeError("attention workspace does not match the launch shape")
    if out is None: out = ws.out if ws.out is not None else torch.empty(B * n_q, D, dtype=q2d.dtype, device=q2d.device)
    if phase == "combine":
        pm, pl, pa = ws.f32_partials()
        _lib.call("gaac_attn_combine", pm, pl, pa, out, B * n_q, nslot, _lib.stream)
        return out
    args = (*_store_args(K), *_store_args(V), q2d, slots, B, n_q, n_kv, SL, S_pad, float(scale), nsplit, K.base3.shape[0],
            kt if has_tail else None, vt if has_tail else None, TL if has_tail else None, TCAP if has_tail else 0)
    if phase == "fused":
        _lib.call("gaac_attn_fused", *args, int(S_all), ws.pm, ws.pl, ws.pa, ws.epoch, out, _lib.stream)
        return out
    args = (*args, *ws.f32_partials())
    if phase == "split":
        _lib.call("gaac_attn_split", *args, _lib.stream)
    else:
        _lib.call("gaac_attn_launch", *args, out, _lib.stream)
    return out


def attention(q, kp, vp, scale=None, nsplit=None, phase="fused"):
    """Decode attention over two Pages (kinds 'k' / 'v', H = B*n_kv heads of equal length).
    q: [B, n_q, D] bf16 (one query token per sequence) -> [B, n_q, D] bf16."""
    B, n_q, Dq = q.shape
    n_kv = kp.H // B
    if nsplit is None: nsplit = launch_nsplit(B, n_kv, kp.S, ragged=False)
    if scale is None: scale = Dq ** -0.5
    if phase == "fused" and Dq == D and 0 < n_q <= GMAX * n_kv and n_q % n_kv == 0:
        out = (_lib._calls or _lib.calls()).attend(kp, vp, n_kv, shared_workspace(B * n_q, nsplit, q.dtype, q.device), q, None, None, kp.sm.shape[1] // D, scale, nsplit,
                                                   None, kp.S, _lib.stream)
        if out is not None: return out
    # the one-kernel launch takes the length as an argument; the other phases read one per head
    SL = None if phase == "fused" else torch.full((kp.H,), kp.S, dtype=torch.int32, device=q.device)
    out = torch.empty(B, n_q, Dq, dtype=q.dtype, device=q.device)
    return attn_launch(kp, vp, q.contiguous(), None, n_q, n_kv, SL, kp.sm.shape[1] // D,
                       scale, nsplit, phase=phase, S_all=kp.S, out=out)


def bf16_attention(q, k, v, scale=None, nsplit=None, ws=None, seq_lens=None, out=None):
    """Baseline: decode attention over UNCOMPRESSED K/V (k, v: [B*n_kv, S, D] bf16, rows contiguous; q: [B, n_q, D]) with the kernel
    structure of the compressed path minus the decoder.  seq_lens: optional int32 [B] device tensor of valid tokens per batch row
    (<= S).  Returns [B, n_q, D] bf16."""
    B, n_q, Dq = q.shape
    H, S, _ = k.shape
    n_kv = H // B
    if k.stride(1) != D or v.stride(1) != D or k.stride(0) != v.stride(0): raise RuntimeError("bf16_attention expects token rows of 128 contiguous elements")
    if nsplit is None: nsplit = choose_nsplit(B, n_kv, S)
    if ws is None: ws = shared_workspace(B * n_q, nsplit, q.dtype, q.device)
    elif ws.rows != B * n_q or ws.nslot != nsplit: raise RuntimeError("attention workspace does not match the launch shape")
    if out is None: out = ws.out if ws.out is not None else torch.empty(B * n_q, D, dtype=q.dtype, device=q.device)
    _lib.call("gaac_bf16_attn", k, v, S, seq_lens, k.stride(0) // D, q.contiguous(), B, n_q, n_kv,
              float(scale if scale is not None else Dq ** -0.5), nsplit, ws.pm, ws.pl, ws.pa, ws.epoch, out, _lib.stream)
    return out.view(B, n_q, Dq)
