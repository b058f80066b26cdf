// Wave-level tile encoder and tile metadata helpers (one wave64 = one 16-token tile), shared by the page encoder,
// the cache append kernel and the paged store.  Tier rule, code words, tag words and escape bytes follow
// /root/reference/gaac/codec.py:138-172 and /root/reference/gaac/encoder.py:30-66; byte placement is the native one
// described in gaac_core.h.
#pragma once
#include "gaac_core.h"

namespace gaac {

// LDS scratch of one encoding wave
constexpr int XROW = D + 8;     // staged row stride in elements: 16 padding bytes spread the sixteen rows of a column over the banks
struct EncodeLds { __align__(16) u16 x[T * XROW]; };     // the tile's BF16 bit patterns, token-major, natural channel order (rows >= nvalid are zero)
// Base words of a head, [0] of the 3-bit tier, [1] of the 4-bit tier: one table for all waves that work on the head
struct BaseTable { u32x4 w[2][NG]; };

// 16 rows of 128 BF16 (row r at src + r*row_stride elements): lane's four 16-byte pieces; rows >= nvalid read as zero (the last valid row is
// loaded in their place: a load under a branch would be waited for by itself).  STREAM: a prompt larger than the caches, read once.
struct RowRegs { u32x4 v[4]; };
template <bool STREAM>
__device__ __forceinline__ void load_rows(RowRegs& R, const u16* __restrict__ src, long row_stride, int nvalid, int lane) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int row = 4 * k + (lane >> 4);
    const u32x4* p = reinterpret_cast<const u32x4*>(src + (long)min(row, nvalid - 1) * row_stride + 8 * (lane & 15));
    R.v[k] = STREAM ? __builtin_nontemporal_load(p) : *p;
  }
  if (nvalid < T) {
#pragma unroll
    for (int k = 0; k < 4; ++k) if (4 * k + (lane >> 4) >= nvalid) R.v[k] = u32x4{0u, 0u, 0u, 0u};
  }
}
__device__ __forceinline__ void store_rows(EncodeLds& L, const RowRegs& R, int lane) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int idx = k * 64 + lane, row = idx >> 4, c16 = idx & 15;
    *reinterpret_cast<u32x4*>(&L.x[row * XROW + c16 * 8]) = R.v[k];
  }
}
// words 2i and 2i + 1 of the table (i < 64)
template <int KIND>
__device__ __forceinline__ u32x2 load_base_pair(const uint8_t* __restrict__ b3row, const uint8_t* __restrict__ b4row, int i) {
  const uint8_t* row = i < 32 ? b3row : b4row;
  const int g = (i >> 1) & 15, p = 2 * (i & 1);
  const u32 l0 = row[chan_of<KIND>(8 * g + p)], h0 = row[chan_of<KIND>(8 * g + p + 4)], l1 = row[chan_of<KIND>(8 * g + p + 1)], h1 = row[chan_of<KIND>(8 * g + p + 5)];
  return u32x2{(l0 << 7) | (h0 << 23), (l1 << 7) | (h1 << 23)};
}

// Orders the LDS traffic of ONE wave (LDS operations of a wave complete in program order; the fences only stop the compiler from
// moving them): what any lane wrote before is visible to every lane of the same wave after.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A word of host memory that the host polls (gaac_wait_words): there before the kernel ends.
__device__ __forceinline__ void store_to_host(int* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM); }

typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
// The encoder works on 32-bit words that hold elements i and i+4 of a unit in their 16-bit halves (the decoder's word order), two
// elements per VALU operation.  The data words of unit u of lane (a, q), and its sign/mantissa bytes (elements 0..3, 4..7):
template <int KIND>
__device__ __forceinline__ void unit_words(const EncodeLds& L, int a, int q, int u, u32* __restrict__ W, u32& slo, u32& shi) {
  u32 l0, h0, l1, h1;      // low and high bytes of elements 0..3 and 4..7
  if (KIND == KIND_K) {
    // elements (2m, 2m+1) are the adjacent channels 32u + 2q + 8m (+1): four aligned words, re-paired to (i, i+4)
    const u32* xr = reinterpret_cast<const u32*>(&L.x[a * XROW + 32 * u + 2 * q]);
    const u32 r0 = xr[0], r1 = xr[4], r2 = xr[8], r3 = xr[12];
    W[0] = __builtin_amdgcn_perm(r2, r0, 0x05040100u); W[1] = __builtin_amdgcn_perm(r2, r0, 0x07060302u);
    W[2] = __builtin_amdgcn_perm(r3, r1, 0x05040100u); W[3] = __builtin_amdgcn_perm(r3, r1, 0x07060302u);
    l0 = __builtin_amdgcn_perm(r1, r0, 0x06040200u); h0 = __builtin_amdgcn_perm(r1, r0, 0x07050301u);
    l1 = __builtin_amdgcn_perm(r3, r2, 0x06040200u); h1 = __builtin_amdgcn_perm(r3, r2, 0x07050301u);
  } else {
    // element i is channel 64 (a & 1) + (a >> 1) + 8 i of token 4q + u
    const u16* xr = &L.x[(4 * q + u) * XROW + 64 * (a & 1) + (a >> 1)];
#pragma unroll
    for (int i = 0; i < 4; ++i) W[i] = __builtin_bit_cast(u32, u16x2_t{xr[8 * i], xr[8 * i + 32]});
    const u32 e0 = __builtin_amdgcn_perm(W[1], W[0], 0x05010400u), e1 = __builtin_amdgcn_perm(W[3], W[2], 0x05010400u);
    const u32 e2 = __builtin_amdgcn_perm(W[1], W[0], 0x07030602u), e3 = __builtin_amdgcn_perm(W[3], W[2], 0x07030602u);
    l0 = __builtin_amdgcn_perm(e1, e0, 0x05040100u); h0 = __builtin_amdgcn_perm(e1, e0, 0x07060302u);
    l1 = __builtin_amdgcn_perm(e3, e2, 0x05040100u); h1 = __builtin_amdgcn_perm(e3, e2, 0x07060302u);
  }
  slo = (l0 & 0x7F7F7F7Fu) | (h0 & 0x80808080u); shi = (l1 & 0x7F7F7F7Fu) | (h1 & 0x80808080u);
}
__device__ __forceinline__ u32 pk_sub_u16(u32 x, u32 y) {
  return __builtin_bit_cast(u32, (u16x2_t)(__builtin_bit_cast(u16x2_t, x) - __builtin_bit_cast(u16x2_t, y)));
}

// What a lane's four units add to the escape stream: tags (2 bits each), the 4th code bits of a 4-bit group (unit u's at byte u; anything where its tag
// is not 1), and where the lane's bytes start among the tile's.
struct UnitEscapes { u32 tag8, eb; int pos; };
// bitwise or across the four 16-lane rows at fixed column
__device__ __forceinline__ u32 quad_rows_or(u32 x) {
  auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  x = r[0] | r[1];
  auto s = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return s[0] | s[1];
}

// ... and their sum
__device__ __forceinline__ u32 quad_rows_add(u32 x) {
  auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  x = r[0] + r[1];
  auto s = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return s[0] + s[1];
}

// Encodes the tile staged in L (after a barrier).  Writes the native sign/mantissa and code bytes and the 16 tag words (one per line); the
// escape bytes stay with the lanes for write_tile_escapes, so that a caller can see their number before it says where they go.
// Returns the tile's escape byte count (all lanes).  Must be called by all 64 lanes of the wave that owns L.  B: the head's base words.
// STREAM: the bytes go past the caches.
// A unit is done with before the next one is read, and what a raw group needs is read again where it is written: 64 registers, so that eight waves share a
// SIMD and hide the trip to memory of a tile's rows (see k_encode_tiles).
template <int KIND, bool STREAM>
__device__ __forceinline__ int encode_staged_tile(const EncodeLds& L, const BaseTable& B, int nvalid, int lane, uint8_t* __restrict__ sm_tile,
                                                  uint8_t* __restrict__ cd_tile, int* __restrict__ flags_tile, UnitEscapes& E) {
  const int a = lane & 15, q = lane >> 4;
  u32 slo[4], shi[4], g24[4];
  E.tag8 = 0u; E.eb = 0u;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    u32 W[4], d3[4], d4[4];
    unit_words<KIND>(L, a, q, u, W, slo[u], shi[u]);
    const u32x4 b3 = B.w[0][unit_group<KIND>(a, q, u)], b4 = B.w[1][unit_group<KIND>(a, q, u)];
#pragma unroll
    for (int i = 0; i < 4; ++i) {      // exponents and their differences at bits 7 and up of the halves: nine bits, negative ones wrap to 257 and more
      W[i] &= EXP_MASK2;
      d3[i] = pk_sub_u16(W[i], b3[i]); d4[i] = pk_sub_u16(W[i], b4[i]);
    }
    // tier rule (codec.py:144-150): all eight differences in 0..7, else all in 0..15, else raw
    const bool fit3 = ((d3[0] | d3[1] | d3[2] | d3[3]) & 0xFC00FC00u) == 0u, fit4 = ((d4[0] | d4[1] | d4[2] | d4[3]) & 0xF800F800u) == 0u;
    u32 c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = fit3 ? d3[i] : (fit4 ? d4[i] : W[i]);
    // code of element i to bits 3i, of element i+4 to 16 + 3i; 4th code bits to 7 + i and 23 + i
    const u32 cacc = ((c[0] >> 7) & 0x00070007u) | ((c[1] >> 4) & 0x00380038u) | ((c[2] >> 1) & 0x01C001C0u) | ((c[3] << 2) & 0x0E000E00u);
    const u32 xacc = ((d4[0] >> 3) & 0x00800080u) | ((d4[1] >> 2) & 0x01000100u) | ((d4[2] >> 1) & 0x02000200u) | (d4[3] & 0x04000400u);
    g24[u] = (cacc & 0xFFFu) | ((cacc >> 4) & ~0xFFFu);
    u32 tag = fit3 ? 0u : (fit4 ? 1u : 3u);
    if (nvalid < T && unit_token<KIND>(a, q, u) >= nvalid) { tag = 0u; g24[u] = 0u; slo[u] = 0u; shi[u] = 0u; }      // padded rows: tier 0, code 0, sign/mantissa 0
    E.tag8 |= tag << (2 * u);
    E.eb |= (((xacc >> 7) & 0xFu) | ((xacc >> 19) & 0xF0u)) << (8 * u);
  }
  u32x4 s0 = {slo[0], shi[0], slo[1], shi[1]}, s1 = {slo[2], shi[2], slo[3], shi[3]};
  const u32 c0 = g24[0] | (g24[1] << 24), c1 = (g24[1] >> 8) | (g24[2] << 16), c2 = (g24[2] >> 16) | (g24[3] << 8);
  u32x4* sm = reinterpret_cast<u32x4*>(sm_tile + 16 * lane); u32* cd = reinterpret_cast<u32*>(cd_tile + 4 * lane);
  if (STREAM) {
    __builtin_nontemporal_store(s0, sm); __builtin_nontemporal_store(s1, sm + 64);
    __builtin_nontemporal_store(c0, cd); __builtin_nontemporal_store(c1, cd + 64); __builtin_nontemporal_store(c2, cd + 128);
  } else { sm[0] = s0; sm[64] = s1; cd[0] = c0; cd[64] = c1; cd[128] = c2; }
  // tag word of line a: this lane owns bits 8q..8q+7 (its four units)
  const u32 f = quad_rows_or(E.tag8 << (8 * q));
  if (lane < T) flags_tile[lane] = (int)f;
  const u32 rb = (u32)esc_bytes(f), incl = row_scan16(rb);
  E.pos = (int)(incl - rb) + esc_prefix(f, 8 * q);
  return __builtin_amdgcn_readlane((int)incl, 15);
}
// The escape bytes of an encoded tile, to esc_tile (the tile's first) on.  L: the tile's rows.
template <int KIND>
__device__ __forceinline__ void write_tile_escapes(const EncodeLds& L, const UnitEscapes& E, uint8_t* esc_tile, int lane) {
  uint8_t* p = esc_tile + E.pos;
  if (__builtin_amdgcn_ballot_w64((E.tag8 & 0xAAu) != 0u) == 0) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if ((E.tag8 >> (2 * u)) & 1u) p[__popc(E.tag8 & ((1u << (2 * u)) - 1u))] = (uint8_t)(E.eb >> (8 * u));
    return;
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const u32 tag = (E.tag8 >> (2 * u)) & 3u;
    if (tag == 1u) p[0] = (uint8_t)(E.eb >> (8 * u));
    else if (tag == 3u) {
      // raw group: the upper five exponent bits of the eight elements, 40 bits little-endian (element i at bit 5i)
      u32 W[4], slo, shi, hl = 0u, hh = 0u;
      unit_words<KIND>(L, lane & 15, lane >> 4, u, W, slo, shi);
#pragma unroll
      for (int i = 0; i < 4; ++i) { hl |= ((W[i] >> 10) & 0x1Fu) << (5 * i); hh |= ((W[i] >> 26) & 0x1Fu) << (5 * i); }
      const u64 h = (u64)hl | ((u64)hh << 20);
#pragma unroll
      for (int k = 0; k < 5; ++k) p[k] = (uint8_t)(h >> (8 * k));
    }
    p += tag_size(tag);
  }
}

// Collects the escape bytes of an encoded tile in LDS, where its rows were.
template <int KIND>
__device__ __forceinline__ const uint8_t* collect_escapes(EncodeLds& L, const UnitEscapes& E, int lane) {
  uint8_t* out = reinterpret_cast<uint8_t*>(L.x);
  uint8_t* p = out + E.pos;
  if (__builtin_amdgcn_ballot_w64((E.tag8 & 0xAAu) != 0u) == 0) {
    wave_lds_sync();      // (every lane has read its units)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if ((E.tag8 >> (2 * u)) & 1u) p[__popc(E.tag8 & ((1u << (2 * u)) - 1u))] = (uint8_t)(E.eb >> (8 * u));
  } else {
    // raw group: the upper five exponent bits of the eight elements, 40 bits little-endian (element i at bit 5i)
    u32 lo[4], hi[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      u32 W[4], slo, shi, hl = 0u, hh = 0u;
      unit_words<KIND>(L, lane & 15, lane >> 4, u, W, slo, shi);
#pragma unroll
      for (int i = 0; i < 4; ++i) { hl |= ((W[i] >> 10) & 0x1Fu) << (5 * i); hh |= ((W[i] >> 26) & 0x1Fu) << (5 * i); }
      lo[u] = hl | (hh << 20); hi[u] = hh >> 12;
    }
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const u32 tag = (E.tag8 >> (2 * u)) & 3u;
      if (tag == 1u) p[0] = (uint8_t)(E.eb >> (8 * u));
      else if (tag == 3u) {
        p[0] = (uint8_t)lo[u]; p[1] = (uint8_t)(lo[u] >> 8); p[2] = (uint8_t)(lo[u] >> 16); p[3] = (uint8_t)(lo[u] >> 24); p[4] = (uint8_t)hi[u];
      }
      p += tag_size(tag);
    }
  }
  wave_lds_sync();
  return out;
}
// Into the worst-case slot of tile `tile` of a head with ntiles, whose 1280 bytes a tile start at slots: the first ESC_HEAD bytes of all tiles lie side by
// side, behind them the rest of each (which a tile in a thousand has), and all of ESC_HEAD is written, whatever of it is used.  Bound by memory: a few bytes
// at the start of every 1280, a partly written line each, were 7 us of a 64K page's 45 without being 1 % of its bytes; now 41.5, and the packing reads
// whole lines.  (Where the bytes go at once, to a stream or a paged slot, write_tile_escapes is as fast without the way through LDS.)
constexpr int ESC_HEAD = 64, ESC_REST = TILE_MAX_ESC - ESC_HEAD;
__device__ __forceinline__ long esc_rest(int tile, int ntiles) { return (long)ntiles * ESC_HEAD + (long)tile * ESC_REST - ESC_HEAD; }      // where byte 0 of the tile would lie
template <int KIND>
__device__ __forceinline__ void write_slot_escapes(EncodeLds& L, const UnitEscapes& E, uint8_t* slots, int tile, int ntiles, int total, int lane) {
  const uint8_t* from = collect_escapes<KIND>(L, E, lane);
  if (lane < ESC_HEAD / 4) reinterpret_cast<u32*>(slots + (long)tile * ESC_HEAD)[lane] = reinterpret_cast<const u32*>(from)[lane];
  for (int i = ESC_HEAD + lane; i < total; i += 64) slots[esc_rest(tile, ntiles) + i] = from[i];
}

// Per-lane metadata of a stored tile: the 2-bit tag of each of the lane's four units and the offset of the unit's escape
// bytes from the start of the tile's escape bytes.  tag_word = the tag word of the lane's line, flags_tile[lane & 15].
struct UnitMeta { u32 tag[4]; int pos[4]; };
__device__ __forceinline__ void tile_unit_meta(u32 tag_word, int lane, UnitMeta& M) {
  const int q = lane >> 4;
  const u32 rb = (u32)esc_bytes(tag_word);
  int pos = (int)(row_scan16(rb) - rb) + esc_prefix(tag_word, 8 * q);
#pragma unroll
  for (int u = 0; u < 4; ++u) { M.tag[u] = (tag_word >> (8 * q + 2 * u)) & 3u; M.pos[u] = pos; pos += tag_size(M.tag[u]); }
}

// Decodes one stored tile (native order) into 16 rows of 128 BF16 in natural channel order: row `tok` at out + tok*row_stride,
// rows >= nvalid are not written.  esc: the tile's escape bytes; b3row / b4row: the 128 base bytes of the head (channel order).
// One wave; bit-exact inverse of encode_staged_tile (codec.py:186-218).
template <int KIND>
__device__ __forceinline__ void decode_tile_rows(const uint8_t* __restrict__ sm_tile, const uint8_t* __restrict__ cd_tile,
                                                 const int* __restrict__ flags_tile, const uint8_t* __restrict__ esc,
                                                 const uint8_t* __restrict__ b3row, const uint8_t* __restrict__ b4row, int lane, int nvalid,
                                                 u16* __restrict__ out, long row_stride) {
  const int a = lane & 15, q = lane >> 4;
  Payload P;
  load_payload(sm_tile, cd_tile, lane, P);
  UnitMeta M;
  tile_unit_meta((u32)flags_tile[a], lane, M);
  u32 b3w[4], b4w[4];
  if (KIND == KIND_V) { load_base_words<KIND>(b3row, a, b3w); load_base_words<KIND>(b4row, a, b4w); }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int tok = unit_token<KIND>(a, q, u), grp = unit_group<KIND>(a, q, u);
    if (KIND == KIND_K) { load_base_words<KIND>(b3row, grp, b3w); load_base_words<KIND>(b4row, grp, b4w); }
    u32 slo, shi, w[4];
    unit_sm(P, u, slo, shi);
    const u32 eb = M.tag[u] == 1u ? (u32)esc[M.pos[u]] : 0u;
    decode_unit(slo, shi, unit_code_word(P.c0, P.c1, P.c2, u), M.tag[u], eb, esc + M.pos[u], b3w, b4w, w);
    if (tok < nvalid) {
      u16* o = out + (long)tok * row_stride;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        o[chan_of<KIND>(8 * grp + p)] = (u16)(w[p] & 0xFFFFu);
        o[chan_of<KIND>(8 * grp + p + 4)] = (u16)(w[p] >> 16);
      }
    }
  }
}

// decode_tile_rows for one wave with LDS of its own, rows 16-byte aligned.  The channel permutation turns the decoder's output into 2-byte
// scattered stores, which LDS absorbs; global memory then gets 16-byte stores, a full 256-byte row per 16 lanes.
//   * The base words of the wave's head lie in LDS, one row per (tier, group), so that the tier select is an address bit (read as bytes
//     from global memory by every lane, they were 64 loads a tile for K and 16 for V).
//   * A lane with at most one raw group has up to eight escape bytes, which lie in the aligned words that hold its first and its last one and
//     the word between: they are loaded at once, without a branch, and no word is touched that holds none of the tile's escape bytes.
//   * K: elements 2m and 2m + 1 of a unit are adjacent channels: one 4-byte LDS store each.  Rows are padded so that the lanes of a store sit in
//     different banks: K's sixteen rows by 16 bytes; V's four rows and two half rows of 64 channels by 32 bytes behind each half.
template <int KIND> struct DecodeLds {
  static constexpr int HALF = KIND == KIND_K ? 64 : 64 + 16, ROW = KIND == KIND_K ? D + 8 : 2 * HALF - 8;      // elements: upper half row, next row
  u32x4 bw[2][NG];
  __align__(16) u16 stage[T * ROW];
};
template <int KIND, bool RAW>      // RAW: some lane of the wave has a raw group
__device__ __forceinline__ void decode_units_to_stage(DecodeLds<KIND>& L, const Payload& P, const u32x4 (&bw)[4], u32 tag8, u32 elo, u32 ehi,
                                                      const uint8_t* __restrict__ esc, int a, int q) {
  // escape byte of unit u at byte u, 0 where its tag is 0: the tags spread to bytes, and their running sum as the selector
  const u32 tb = ((tag8 & 0x55u) * 0x41041u) & 0x01010101u, sel = (tb << 8) + (tb << 16) + (tb << 24);
  const u32 eb4 = __builtin_amdgcn_perm(0u, elo, sel) & ((tb << 8) - tb);
  const bool lane_raw = (tag8 & 0xAAu) != 0u, lane_raws = __popc(tag8 & 0xAAu) > 1;
  u32 off = 0u;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const u32 tag = (tag8 >> (2 * u)) & 3u;
    u32 eb = (eb4 >> (8 * u)) & 0xFFu, hi = 0u;
    if (RAW) {      // behind or at a raw group: one byte, or the five of the group, from `off` on
      u64 v = ((u64)elo | ((u64)ehi << 32)) >> (8u * (off & 7u));
      if (lane_raws && tag) {      // beyond the bytes at hand: the aligned words of the first and the last one
        const uintptr_t p = reinterpret_cast<uintptr_t>(esc) + off;
        const u64 w = (u64)*reinterpret_cast<const u32*>(p & ~(uintptr_t)3) | ((u64)*reinterpret_cast<const u32*>((p + (tag == 3u ? 4 : 0)) & ~(uintptr_t)3) << 32);
        v = w >> (8u * (u32)(p & 3));
      }
      eb = lane_raw ? (tag ? (u32)v & 0xFFu : 0u) : eb;
      eb = tag == 3u ? (u32)v : eb; hi = (u32)(v >> 32);
      off += (u32)tag_size(tag);
    }
    u32x4 x;
    const u32 xw = eb | (eb << 12);      // 4th code bits: element i at bit i, element i + 4 at bit 16 + i
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = (xw << (10 - i)) & 0x04000400u;
    if (RAW) {
      const u32x4 xr = raw_x_words(eb, hi, bw[u]);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = tag == 3u ? xr[i] : x[i];
    }
    u32 slo, shi, w[4];
    unit_sm(P, u, slo, shi);
    decode_unit_x(slo, shi, unit_code_word(P.c0, P.c1, P.c2, u), x, bw[u], w);
    if (KIND == KIND_K) {
      u32* row = reinterpret_cast<u32*>(L.stage + a * DecodeLds<KIND>::ROW) + 16 * u + q;      // channels 32u + 2q + 8m, + 1
      row[0] = __builtin_amdgcn_perm(w[1], w[0], 0x05040100u); row[4] = __builtin_amdgcn_perm(w[3], w[2], 0x05040100u);
      row[8] = __builtin_amdgcn_perm(w[1], w[0], 0x07060302u); row[12] = __builtin_amdgcn_perm(w[3], w[2], 0x07060302u);
    } else {
      u16* row = L.stage + (4 * q + u) * DecodeLds<KIND>::ROW + DecodeLds<KIND>::HALF * (a & 1) + (a >> 1);      // channel 64 (a & 1) + (a >> 1) + 8i
#pragma unroll
      for (int i = 0; i < 4; ++i) { row[8 * i] = (u16)w[i]; row[8 * i + 32] = (u16)(w[i] >> 16); }
    }
  }
}
template <int KIND>
__device__ __forceinline__ void decode_tile_staged(const uint8_t* __restrict__ sm_tile, const uint8_t* __restrict__ cd_tile,
                                                   const int* __restrict__ flags_tile, const uint8_t* __restrict__ esc,
                                                   const uint8_t* __restrict__ b3row, const uint8_t* __restrict__ b4row, int lane, int nvalid,
                                                   DecodeLds<KIND>& L, u16* __restrict__ out, long row_stride) {
  const int a = lane & 15, q = lane >> 4;
  const u32 f = (u32)flags_tile[a];
  const u32x2 base_pair = load_base_pair<KIND>(b3row, b4row, lane);
  Payload P;
  load_payload<false>(sm_tile, cd_tile, lane, P);
  const u32 rb = (u32)esc_bytes(f), tag8 = __builtin_amdgcn_ubfe(f, 8 * q, 8);
  esc += row_scan16(rb) - rb + (u32)esc_prefix(f, 8 * q);
  const int nb = esc_bytes(tag8);
  // (no escapes: any word that is there)
  const uintptr_t e0 = nb ? reinterpret_cast<uintptr_t>(esc) : reinterpret_cast<uintptr_t>(flags_tile), ea = e0 & ~(uintptr_t)3, ez = (e0 + max(nb - 1, 0)) & ~(uintptr_t)3;
  const u32 w0 = *reinterpret_cast<const u32*>(ea), w1 = *reinterpret_cast<const u32*>(min(ea + 4, ez)), w2 = *reinterpret_cast<const u32*>(ez);
  reinterpret_cast<u32x2*>(&L.bw[0][0])[lane] = base_pair;
  wave_lds_sync();
  u32x4 bw[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) bw[u] = L.bw[(tag8 >> (2 * u)) & 1u][unit_group<KIND>(a, q, u)];
  const u32 elo = __builtin_amdgcn_alignbyte(w1, w0, (u32)e0 & 3u), ehi = __builtin_amdgcn_alignbyte(w2, w1, (u32)e0 & 3u);
  if (__builtin_amdgcn_ballot_w64((tag8 & 0xAAu) != 0u) == 0) decode_units_to_stage<KIND, false>(L, P, bw, tag8, elo, ehi, esc, a, q);
  else decode_units_to_stage<KIND, true>(L, P, bw, tag8, elo, ehi, esc, a, q);
  wave_lds_sync();
  // The rows go past the caches, the tile through them (the other way round from the attention's stream): 8 x 65536 tokens 44 -> 41.5 us
  // with such stores, 8 x 16384 14.4 -> 13.8, and 11.8 with loads that find the tile in the Infinity Cache
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int idx = k * 64 + lane, row = idx >> 4, c16 = idx & 15;
    const u32x4 v = *reinterpret_cast<const u32x4*>(L.stage + row * DecodeLds<KIND>::ROW + c16 * 8 + (c16 >= 8 ? DecodeLds<KIND>::HALF - 64 : 0));
    if (row < nvalid) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out + (long)row * row_stride + c16 * 8));
  }
}

}  // namespace gaac
