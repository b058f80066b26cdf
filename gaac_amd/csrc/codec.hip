// Calibration, page encoder and page decoder kernels + their extern "C" entry points.
//   exponent_hist / bases_from_hist   /root/reference/gaac/codec.py:70-84
//   encode_tiles / compact            /root/reference/gaac/encoder.py:16-76, 94-109
//   row_offsets                       /root/reference/gaac/codec.py:221-225
//   decode_tiles                      /root/reference/gaac/codec.py:186-218
#include <algorithm>
#include <chrono>
#include "gaac_tile.h"
#include "gaac_capi.h"
#include "../../include/gaac_hip.h"

namespace gaac {

char* last_error_buffer() { static thread_local char buf[512] = {0}; return buf; }

// ---------------------------------------------------------------------------------------------------- calibration
// Exponent histogram per (kv head, channel).  A block owns the 128 channels of one kv head of K or of V and a chunk of tokens.  A lane
// of every wave counts two adjacent channels of a row in a table of 256 x 64 words that the block's waves share: word (bin, lane) holds the counts of
// the two in its 16-bit halves (a chunk has at most 65535 tokens), so a lane only ever touches its own bank and the LDS adds of a wave never collide,
// however alike the exponents are.  (A table of one word per (channel, bin) with eight lanes to a row sent all rows of a wave to the same
// few words of a channel and took twice as long.)  A load takes four rows, 16 bytes a lane; sixteen lanes of a row each hold four words, and two lane
// exchanges give every lane one word of all four rows.
// Bound by the reads (without counting at all: 29 us with the launch).  K and V of 32768 tokens x 8 kv heads, 134 MB: 27.3 us = 4.9 TB/s; eight waves that read
// 4 bytes a lane, sixteen rows at a time, 28.4 with whole batches and 33 with the rest of a chunk row by row: a prompt of 30011 tokens 90.2 us a call
// -> 86.6, of 12345 62.7 -> 57.3, of 4000 44.2 -> 40.3, of 32768 91.3 -> 90.4.  More loads in flight are slower: 28.2 with three, 27.9 with eight.
// PARTS = false: the non-zero counts are added to 64-bit ones at the end, hist[row][256], the layout that gaac_exponent_hist hands out.  PARTS = true: a block leaves
// its own table, the rows (bins) of it that hold a count, and a bit for each of these; k_prompt_bases adds up the blocks' tables.  Added to one global table,
// which a launch had to clear first, the counts of a prompt took that launch longer: 32768 tokens x 8 heads 88.1 -> 83.2 us a call, 4000 tokens 26.2 -> 24.5 of
// kernels.
constexpr int HIST_WAVES = 16, HIST_MAX_CHUNK = 65535, HIST_LOADS = 2, HIST_TABLES = 64;      // HIST_LOADS: loads of four rows in flight per wave
constexpr long HIST_TABLE = 256 * 64 * sizeof(u32) + HIST_WAVES * sizeof(u16);      // bytes
struct HistArgs { const u16* x[2]; long head_stride[2], row_stride[2]; long n_tok; int chunk, n_kv; unsigned long long* hist; u32* rows; u16* bits; };      // rows [pair][chunk][256][64], bits [pair][chunk][16]
template <bool PARTS>
__global__ void __launch_bounds__(64 * HIST_WAVES) k_exponent_hist(const HistArgs A) {
  __shared__ u32 h[256 * 64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, head = blockIdx.y, kind = blockIdx.z;
  const long t0 = (long)blockIdx.x * A.chunk, t1 = min(t0 + (long)A.chunk, A.n_tok);
  const long rs = A.row_stride[kind];
  const u16* xp = A.x[kind] + (long)head * A.head_stride[kind] + 8 * (lane & 15);
  u32* hc = h + lane;
  const auto count = [&](u32 w) {
    atomicAdd(&hc[((w >> 7) & 0xFFu) << 6], 1u);
    atomicAdd(&hc[((w >> 23) & 0xFFu) << 6], 0x10000u);
  };
  // Rows of the chunk: a load of the wave takes four, 4 HIST_WAVES further on than the one before; each is repeated for the next round as soon as its
  // rows are counted.  Rows past the end read the last one (no load under a branch) and are not counted.
  const int n = (int)(t1 - t0), r0 = 4 * __builtin_amdgcn_readfirstlane(wave);
  const u16* x0 = xp + t0 * rs;
  const auto load = [&](int r) { return load_u32x4_unaligned(x0 + (long)min(r + (lane >> 4), n - 1) * rs); };
  u32x4 w[HIST_LOADS];
#pragma unroll
  for (int k = 0; k < HIST_LOADS; ++k) w[k] = load(r0 + 4 * HIST_WAVES * k);
  for (int i = tid; i < 256 * 64 / 4; i += 64 * HIST_WAVES) reinterpret_cast<u32x4*>(h)[i] = u32x4{0u, 0u, 0u, 0u};
  __syncthreads();
  for (int r = r0; r < n; r += 4 * HIST_WAVES * HIST_LOADS) {
#pragma unroll
    for (int k = 0; k < HIST_LOADS; ++k) {
      // lane (q, c) = (lane >> 4, lane & 15) has words 4c .. 4c + 3 of row q; after the exchange it has word 4c + q of all four rows
      u32 x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = (u32)__builtin_amdgcn_mov_dpp((int)w[k][j], 0xE4 /* quad_perm: in place */, 0xF, 0xF, true);      // (a copy: exchanged in place, the loop's end waits for all loads)
      const auto a = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false), b = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
      const auto lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
      const int row = r + 4 * HIST_WAVES * k;
      w[k] = load(row + 4 * HIST_WAVES * HIST_LOADS);
      if (row + 3 < n) { count(lo[0]); count(lo[1]); count(hi[0]); count(hi[1]); }
      else {
        if (row < n) count(lo[0]);
        if (row + 1 < n) count(lo[1]);
        if (row + 2 < n) count(hi[0]);
      }
    }
  }
  __syncthreads();
  const long pair = (long)kind * A.n_kv + head;
  const int word = 4 * (lane & 15) + (lane >> 4);      // of the row, that the lane counted
  if (PARTS) {
    constexpr int BINS = 256 / HIST_WAVES;      // a wave's, every sixteenth: the ones in use lie side by side
    const long at = pair * gridDim.x + blockIdx.x;
    u32* rows = A.rows + at * (256 * 64);
    u32 c[BINS], bits = 0u;
#pragma unroll
    for (int i = 0; i < BINS; ++i) c[i] = h[64 * (wave + HIST_WAVES * i) + lane];
#pragma unroll
    for (int i = 0; i < BINS; ++i)
      if (__builtin_amdgcn_ballot_w64(c[i] != 0u) != 0) { rows[64 * (wave + HIST_WAVES * i) + word] = c[i]; bits |= 1u << i; }
    if (lane == 0) A.bits[at * HIST_WAVES + wave] = (u16)bits;
    return;
  }
  for (int i = tid; i < 256 * 64; i += 64 * HIST_WAVES) {
    const u32 c = h[i];
    if (c == 0u) continue;
    unsigned long long* row = A.hist + (pair * D + 2 * word) * 256 + (i >> 6);
    if (c & 0xFFFFu) atomicAdd(row, (unsigned long long)(c & 0xFFFFu));
    if (c >> 16) atomicAdd(row + 256, (unsigned long long)(c >> 16));
  }
}
static int hist_chunks(long n_tok, int pairs, bool parts) {
  // one block per CU, at least 256 tokens each, so that clearing and scanning the 64 KB table stays the smaller part (two blocks per CU,
  // which the LDS has room for: 26 against 23.6 us for 2 x 8 heads x 32768 tokens out of the Infinity Cache, measured with blocks of eight waves)
  // (tables that another launch adds up: no more than HIST_TABLES of a (kind, head).  32768 tokens x 1 head, 128 / 64 tables: histogram 5.7 / 6.3 us, bases 12.4 / 8.0,
  // the call 39.1 / 36.4)
  const long n = min((n_tok + 255) / 256, (long)min(max(1, 256 / pairs), parts ? HIST_TABLES : 256));
  return (int)max(n, (n_tok + HIST_MAX_CHUNK - 1) / HIST_MAX_CHUNK);
}
static int launch_hist(HistArgs& A, int kinds, int nchunk, hipStream_t stream) {      // returns the blocks of a (kind, head), nchunk at most
  A.chunk = (int)((A.n_tok + nchunk - 1) / nchunk);
  const dim3 grid((unsigned)((A.n_tok + A.chunk - 1) / A.chunk), A.n_kv, kinds);
  if (A.rows) hipLaunchKernelGGL(k_exponent_hist<true>, grid, dim3(64 * HIST_WAVES), 0, stream, A);
  else hipLaunchKernelGGL(k_exponent_hist<false>, grid, dim3(64 * HIST_WAVES), 0, stream, A);
  return (int)grid.x;
}

// The bases of K and V of a prompt from the tables of its k_exponent_hist<true>, written to base row row0 + head of the two kinds' tables.  A block takes 32 channels
// of one (kind, head): a wave adds up every sixteenth row over the tables, the 256 sums of a channel go to LDS, thread (channel, eighth) slides the two windows over
// 32 starts.  Latency: two trips to memory, bits and rows, if a lane has R loads of a row in flight for up to 4 R tables: with four for any number of them, sixteen
// tables a trip, 32768 tokens x 1 head (128 tables) took 14.2 us, x 2 (64) 8.6, x 4 (32) 5.8; now, with 64 at most, 8.0, 7.4 and 5.1 (x 8, 16 tables, 4.7).  (A table a
// wave and LDS atomics for the sums: 6.4 us instead of 4.8.)
struct PromptBasesArgs { const u32* rows; const u16* bits; int chunks; uint8_t* b3[2]; uint8_t* b4[2]; int n_kv, row0; };
template <int R>
__global__ void __launch_bounds__(1024) k_prompt_bases(const PromptBasesArgs A) {
  constexpr int STRIDE = 256 + 17;      // odd: the 32 channels of a bin sit in different banks
  __shared__ u32 cnt[32 * STRIDE];
  __shared__ u32 best[2][8][32];
  __shared__ int arg[2][8][32];
  const int tid = threadIdx.x, grp = blockIdx.x, head = blockIdx.y, kind = blockIdx.z;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const long at0 = ((long)kind * A.n_kv + head) * A.chunks;
  const u16* bits = A.bits + at0 * HIST_WAVES + wave;
  const u32* words = A.rows + at0 * (256 * 64) + 64 * wave + 16 * grp;
  u32* sums = cnt + 2 * (lane & 15) * STRIDE + wave;
  // lane (j, w): word w of the channels' sixteen, of the tables c0 + j, c0 + 4 + j, ...; the next tables' bits are on their way meanwhile
  const auto table = [&](int c0, int r) { return c0 + 4 * r + (lane >> 4); };
  u32 next[R];
  if (A.chunks > 0)      // (an empty prompt has no tables)
#pragma unroll
    for (int r = 0; r < R; ++r) next[r] = bits[(u32)min(table(0, r), A.chunks - 1) * HIST_WAVES];
  for (int i = tid; i < 32 * STRIDE; i += 1024) cnt[i] = 0u;
  __syncthreads();
  for (int c0 = 0; c0 < A.chunks; c0 += 4 * R) {
    u32 has[R], at[R], any = 0u;
#pragma unroll
    for (int r = 0; r < R; ++r) { has[r] = table(c0, r) < A.chunks ? next[r] : 0u; any |= has[r]; }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      at[r] = (u32)min(table(c0, r), A.chunks - 1) * (256 * 64) + (u32)(lane & 15);
      next[r] = bits[(u32)min(table(c0 + 4 * R, r), A.chunks - 1) * HIST_WAVES];
    }
    u32 left = __builtin_amdgcn_readfirstlane(quad_rows_or(any));
    while (left) {      // two rows at a time, R tables a lane
      const int i0 = __builtin_ctz(left);
      left &= left - 1;
      const int i1 = left ? __builtin_ctz(left) : i0;
      const u32 *w0 = words + 64 * HIST_WAVES * i0, *w1 = words + 64 * HIST_WAVES * i1;
      u32 v0[R], v1[R], lo0 = 0u, hi0 = 0u, lo1 = 0u, hi1 = 0u;
#pragma unroll
      for (int r = 0; r < R; ++r) { v0[r] = w0[at[r]]; v1[r] = w1[at[r]]; }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        v0[r] = (has[r] >> i0) & 1u ? v0[r] : 0u; v1[r] = (has[r] >> i1) & 1u ? v1[r] : 0u;      // (a row without the bit holds anything)
        lo0 += v0[r] & 0xFFFFu; hi0 += v0[r] >> 16; lo1 += v1[r] & 0xFFFFu; hi1 += v1[r] >> 16;
      }
      lo0 = quad_rows_add(lo0); hi0 = quad_rows_add(hi0); lo1 = quad_rows_add(lo1); hi1 = quad_rows_add(hi1);
      if (lane < 16) {
        sums[HIST_WAVES * i0] += lo0; sums[STRIDE + HIST_WAVES * i0] += hi0;
        if (left) { sums[HIST_WAVES * i1] += lo1; sums[STRIDE + HIST_WAVES * i1] += hi1; }
      }
      left &= left - 1;
    }
  }
  __syncthreads();
  const int c = tid & 31, part = (tid >> 5) & 7, st0 = 32 * part;
  if (tid < 256) {
  u32 n[32 + 15];      // the counts that the thread's windows cover, read together
#pragma unroll
  for (int i = 0; i < 32 + 15; ++i) n[i] = cnt[c * STRIDE + min(st0 + i, 255)];
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int win = pass ? 16 : 8;
    u32 sum = 0u;
#pragma unroll
    for (int i = 0; i < win; ++i) sum += n[i];
    u32 b = sum; int a = st0;
#pragma unroll
    for (int i = 1; i < 32; ++i) {      // the lowest start of the largest sum, as k_bases_from_hist
      sum += n[i + win - 1] - n[i - 1];
      if (st0 + i + win <= 256 && sum > b) { b = sum; a = st0 + i; }
    }
    best[pass][part][c] = b; arg[pass][part][c] = a;
  }
  }
  __syncthreads();
  if (tid < 64) {
    const int pass = tid >> 5;
    u32 b = best[pass][0][c]; int a = arg[pass][0][c];
#pragma unroll
    for (int p = 1; p < 8; ++p) if (best[pass][p][c] > b) { b = best[pass][p][c]; a = arg[pass][p][c]; }
    (pass ? A.b4[kind] : A.b3[kind])[(long)(A.row0 + head) * D + 32 * grp + c] = (uint8_t)a;
  }
}

// One wave per histogram row: lane l evaluates the windows that start at 4l .. 4l+3 (the reference takes the first maximum of the
// window sums, codec.py:70-77: the lowest start wins ties).
__global__ void __launch_bounds__(256) k_bases_from_hist(const long long* __restrict__ hist, int rows,
                                                         uint8_t* __restrict__ base3, uint8_t* __restrict__ base4) {
  __shared__ long long hs[4][256 + 16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = blockIdx.x * 4 + wave;
  if (r >= rows) return;
  long long* hr = hs[wave];
#pragma unroll
  for (int k = 0; k < 4; ++k) hr[lane + 64 * k] = hist[(long)r * 256 + lane + 64 * k];
  if (lane < 16) hr[256 + lane] = 0;
  wave_lds_sync();
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int w = pass ? 16 : 8;
    long long best = -1; int arg = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int st = 4 * lane + j;
      long long sum = 0;
      for (int i = 0; i < w; ++i) sum += hr[st + i];
      if (st + w <= 256 && sum > best) { best = sum; arg = st; }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {      // maximum, lowest start among equals
      const long long ob = __shfl_xor(best, o, 64); const int oa = __shfl_xor(arg, o, 64);
      if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
    }
    if (lane == 0) (pass ? base4 : base3)[r] = (uint8_t)arg;
  }
}

// ---------------------------------------------------------------------------------------------------- page encoder
// A block of four waves takes four consecutive tiles of one head, one each (one-wave blocks would be limited by the rate at which workgroups can be
// launched), and makes the head's base words for all of them.  K and V of a prompt share a launch (blockIdx.z): one start-up and one drain for both.
// Bound by the memory rate.  A wave has one tile and 62 registers: eight waves a SIMD hide each other's trips to memory.  Before, a wave took four tiles in
// a row with the rows of the next one and all base words in registers, 147 of them: three waves a SIMD and a quarter more instructions a tile; 64K page of 8 heads
// out of memory 47.9 -> 45.0 us (with the slots of write_slot_escapes 41.5: 229 MB, 5.5 TB/s), 16K page 15.9 -> 14.6 (13.4), prompt of 32768 tokens with given bases 49.1 -> 46.6.
// What goes past the caches is chosen by what comes next, so that the Infinity Cache keeps the rest:
//   * the rows of a large launch (BIG) are read for the last time: 64K page 44.6 -> 42.3 us; the 32768-token prompt's call, where the histogram has
//     just brought them in, 109 -> 101 us;
//   * a prompt's tiles (PROMPT) are stored past them, or they would push out rows that are still to be read: 119 -> 109 us; a page's are not,
//     the caller is as likely to read them at once: 64K page and back 107 us past the caches, 101 through them.
constexpr int CODEC_WAVES = 4;
struct EncodeKind {      // one of K, V
  const u16* x; long head_stride, row_stride;
  const uint8_t* b3; const uint8_t* b4;
  uint8_t* sm; uint8_t* cd; int* flags;            // head 0 of the call; token stride S_pad
  uint8_t* slots; int* tile_bytes;                 // [H][ntiles] worst-case escape slots and the bytes used in each
};
struct EncodeArgs { EncodeKind k, v; int kind0, S, S_pad, ntiles, brow0, NB; const int* bidx; };      // blockIdx.z = 0 is kind0
struct EncodeBlockLds { BaseTable B; EncodeLds w[CODEC_WAVES]; };
template <int KIND, bool BIG, bool PROMPT>
__device__ __forceinline__ void encode_tiles_body(const EncodeArgs& A, const EncodeKind& J, EncodeBlockLds& L, int h, int tile, int wave, int lane) {
  const int S = A.S, ntiles = A.ntiles, nvalid = min(T, S - tile * T);
  const int brow = A.bidx ? A.bidx[h] : (A.brow0 + h) % A.NB;
  RowRegs R;
  load_rows<BIG>(R, J.x + (long)h * J.head_stride + (long)min(tile, ntiles - 1) * T * J.row_stride, J.row_stride, max(nvalid, 1), lane);
  if (wave == 0) reinterpret_cast<u32x2*>(&L.B.w[0][0])[lane] = load_base_pair<KIND>(J.b3 + (long)brow * D, J.b4 + (long)brow * D, lane);
  store_rows(L.w[wave], R, lane);
  __syncthreads();
  if (tile >= ntiles) return;
  const long row0 = (long)h * A.S_pad + (long)tile * T;
  UnitEscapes E;
  const int total = encode_staged_tile<KIND, PROMPT>(L.w[wave], L.B, nvalid, lane, J.sm + row0 * D, J.cd + row0 * CB, J.flags + row0, E);
  write_slot_escapes<KIND>(L.w[wave], E, J.slots + (long)h * ntiles * TILE_MAX_ESC, tile, ntiles, total, lane);
  if (lane == 0) J.tile_bytes[(long)h * ntiles + tile] = total;
}
template <bool BIG, bool PROMPT>
__global__ void __launch_bounds__(64 * CODEC_WAVES, 8) k_encode_tiles(const EncodeArgs A) {
  __shared__ EncodeBlockLds L;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, tile = blockIdx.x * CODEC_WAVES + wave;
  if (A.kind0 + (int)blockIdx.z == KIND_K) encode_tiles_body<KIND_K, BIG, PROMPT>(A, A.k, L, blockIdx.y, tile, wave, lane);
  else encode_tiles_body<KIND_V, BIG, PROMPT>(A, A.v, L, blockIdx.y, tile, wave, lane);
}
template <bool PROMPT>
static void launch_encode(const EncodeArgs& A, int H, int kinds, hipStream_t stream) {
  const dim3 grid((A.ntiles + CODEC_WAVES - 1) / CODEC_WAVES, H, kinds);
  if ((long)A.ntiles * H * kinds >= 8192) hipLaunchKernelGGL((k_encode_tiles<true, PROMPT>), grid, dim3(64 * CODEC_WAVES), 0, stream, A);
  else hipLaunchKernelGGL((k_encode_tiles<false, PROMPT>), grid, dim3(64 * CODEC_WAVES), 0, stream, A);
}

// Exclusive prefix sums of one head's tile sizes into off, and their total; called by all threads of a block, of which each SCAN_NT
// scan one list (tid: the thread's index among these; sh: one int per wave of the list).
// Latency: a chain of load, scan, exchange between the waves, store.  A thread that took eight tiles in a row touched a line per lane in each
// of its loads and stores: 5.4 us for 8 x 4096 tiles with k_tile_scan, 6.4 with k_prompt_scan; lane by lane 4.3 and 4.9.
constexpr int SCAN_NT = 512, SCAN_PER = 8;
__device__ __forceinline__ int scan_tile_bytes(const int* __restrict__ tb, int* __restrict__ off, int ntiles, int tid, int* sh) {
  const int wave = tid >> 6, lane = tid & 63;
  int carry = 0;
  for (int base = 0; base < ntiles; base += SCAN_NT * SCAN_PER) {
    const int t0 = base + wave * (64 * SCAN_PER) + lane;      // the wave's tiles t0, t0 + 64, ...: whole lines in every load and store
    int n[SCAN_PER], incl[SCAN_PER], mine = 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k) n[k] = tb[min(t0 + 64 * k, ntiles - 1)];
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k) {
      n[k] = t0 + 64 * k < ntiles ? n[k] : 0;
      const int x = (int)row_scan16((u32)n[k]), r0 = __builtin_amdgcn_readlane(x, 15), r1 = __builtin_amdgcn_readlane(x, 31), r2 = __builtin_amdgcn_readlane(x, 47);
      incl[k] = mine + x + (lane >= 16 ? r0 : 0) + (lane >= 32 ? r1 : 0) + (lane >= 48 ? r2 : 0);
      mine += r0 + r1 + r2 + __builtin_amdgcn_readlane(x, 63);
    }
    if (lane == 0) sh[wave] = mine;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < SCAN_NT / 64; ++w) { const int v = sh[w]; all += v; before += w < wave ? v : 0; }
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k) if (t0 + 64 * k < ntiles) off[t0 + 64 * k] = carry + before + incl[k] - n[k];
    carry = carry > 0x7FFFFFFF - all ? 0x7FFFFFFF : carry + all;      // (all: at most 4096 tiles of 1280 bytes)
    __syncthreads();
  }
  return carry;
}
// Tile offsets and escape totals of the heads, one block per head.  host_bytes (or null): the totals once more in host memory that the
// device can write, for the caller that sizes the stream: it spares a copy and its latency.
__global__ void __launch_bounds__(SCAN_NT) k_tile_scan(const int* __restrict__ tile_bytes, int* __restrict__ tile_off, int ntiles,
                                                       int* __restrict__ head_bytes, int* __restrict__ host_bytes) {
  __shared__ int sh[SCAN_NT / 64];
  const long h = blockIdx.x;
  const int total = scan_tile_bytes(tile_bytes + h * ntiles, tile_off + h * ntiles, ntiles, threadIdx.x, sh);
  if (threadIdx.x == 0) {
    if (head_bytes) head_bytes[h] = total;
    if (host_bytes) store_to_host(host_bytes + h, total);
  }
}

// Packs the per-tile escape slots into the heads' streams.  A block takes 64 consecutive tiles of a head, a wave 16 of them: the sizes and
// offsets of its tiles in one load each, then the first 64 bytes of all 16 slots in flight together (a tile has about 30 escape bytes;
// what is beyond 64 follows in a loop).  A wave that copied its tiles one after the other, each a chain of size -> bytes -> store, took
// 20.7 us for the 8 x 4096 tiles of a 64K-token page; this one takes 6.6 us and writes the row offsets as well (9.2 us of their own before).
// HEADS: the streams lie back to back and the block derives its head's start from the totals of the heads (a Page; it also
// writes head_start, the row offsets and the stream's padding); else head_start is given and a head whose window is too small is left out.
constexpr int PACK_TPB = 64;
struct PackKind { const uint8_t* slots; const int* tile_bytes; const int* tile_off; long off_stride; const int* head_start; uint8_t* ovf; };
struct PackArgs {
  PackKind j[2]; int ntiles;
  const int* head_bytes;                 // [kinds * H] totals (null without HEADS: every window is large enough)
  int window;                            // bytes that a head's stream must fit in (without HEADS)
  long ovf_cap;                          // bytes there are for all streams and the padding: where they are too few, none is written (HEADS)
  const int* flags; int S, S_pad; int* head_start_out; int* ovf_off;      // HEADS
};
template <bool HEADS>
__global__ void __launch_bounds__(256) k_pack(const PackArgs A) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.y, H = gridDim.y;
  const PackKind& J = A.j[blockIdx.z];
  const int t0 = blockIdx.x * PACK_TPB + 16 * wave, n_own = min(16, A.ntiles - t0);      // (may be <= 0)
  const int tl = min(t0 + (lane & 15), A.ntiles - 1);
  const int nb = J.tile_bytes[(long)h * A.ntiles + tl], of = J.tile_off[(long)h * J.off_stride + tl];
  const uint8_t* src = J.slots + (long)h * A.ntiles * TILE_MAX_ESC;
  u32 v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = src[(long)min(t0 + k, A.ntiles - 1) * ESC_HEAD + lane];
  long start = 0;
  bool fits = true;
  if (HEADS) {
    __shared__ long part[2][4];
    long before = 0, all = 0;
    for (int i = tid; i < H; i += 256) { const int n = A.head_bytes[i]; all += n; before += i < h ? n : 0; }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { before += __shfl_xor(before, o, 64); all += __shfl_xor(all, o, 64); }
    if (lane == 0) { part[0][wave] = before; part[1][wave] = all; }
    __syncthreads();
    start = (part[0][0] + part[0][1]) + (part[0][2] + part[0][3]); all = (part[1][0] + part[1][1]) + (part[1][2] + part[1][3]);
    fits = all < 0x7FFFFFFF && all + 8 <= A.ovf_cap;      // (a head's total stops at 2^31 - 1)
    if (blockIdx.x == 0 && tid == 0) {
      A.head_start_out[h] = (int)start;
      if (h == H - 1) A.head_start_out[H] = (int)all;
    }
    if (fits && blockIdx.x == 0 && h == H - 1 && tid < 8) J.ovf[all + tid] = 0;      // readers fetch eight bytes at a time
  } else {
    if (A.head_bytes && A.head_bytes[(long)blockIdx.z * H + h] > A.window) return;
    start = J.head_start[h];
  }
  uint8_t* dst = J.ovf + start;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int n = __builtin_amdgcn_readlane(nb, k), o = __builtin_amdgcn_readlane(of, k);
    if (k >= n_own || !fits) break;
    if (lane < n) dst[o + lane] = (uint8_t)v[k];
    for (int i = 64 + lane; i < n; i += 64) dst[o + i] = src[esc_rest(t0 + k, A.ntiles) + i];
  }
  if (HEADS) {      // row offsets: tile offset + the escape bytes of the tile's earlier tag words
    const int* fl = A.flags + (long)h * A.S_pad;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = t0 * T + 64 * k + lane;
      const u32 rb = (u32)esc_bytes((u32)fl[min(i, A.S_pad - 1)]), incl = row_scan16(rb);
      const int to = __shfl(of, 4 * k + (lane >> 4), 64);
      if (i < A.S && n_own > 0) A.ovf_off[(long)h * A.S + i] = to + (int)(incl - rb);
    }
  }
}

// k_tile_scan and k_pack<HEADS> in one launch, for pages of up to PAGE_PACK_TILES tiles over all heads: a block of 64 tiles adds up the sizes of all
// tiles, of the heads before its own and of the tiles before its own by itself (PER loads a thread in flight, from the L2).  Latency, like the two.
// In a graph, us, one launch against two: 2048 tiles 5.4 / 7.9, 8192 6.1 / 8.0, 16384 7.6 / 8.1, 32768 13.7 / 8.7 (every block reads every size).
// It and the two others are launched without a look at the totals by the host, which sees them while the slots are packed:
// 8 x 4096 tokens encoded and expanded again 45.2 -> 37.9 us a call, 8 x 65536 100.0 -> 90.4.
constexpr int PAGE_PACK_TILES = 16384;
struct PagePackArgs {
  const uint8_t* slots; const int* tile_bytes; int* tile_off; int* head_bytes; int* host_bytes; int ntiles;
  const int* flags; int S, S_pad; int* head_start; uint8_t* ovf; long ovf_cap; int* ovf_off;
};
__global__ void __launch_bounds__(256) k_page_pack(const PagePackArgs A) {
  constexpr int PER = 16;
  __shared__ u32x4 part[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.y, H = gridDim.y, ntiles = A.ntiles;
  const int tile0 = blockIdx.x * PACK_TPB, t0 = tile0 + 16 * wave, n_own = min(16, ntiles - t0);      // (n_own may be <= 0)
  const int head0 = h * ntiles, own0 = head0 + tile0, all_tiles = H * ntiles;
  // every load up front, none under a branch
  const uint8_t* src = A.slots + (long)head0 * TILE_MAX_ESC;
  int n = A.tile_bytes[head0 + min(tile0 + lane, ntiles - 1)];
  u32 v[16], fl[4];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = src[(long)min(t0 + k, ntiles - 1) * ESC_HEAD + lane];
#pragma unroll
  for (int k = 0; k < 4; ++k) fl[k] = (u32)A.flags[(long)h * A.S_pad + min(t0 * T + 64 * k + lane, A.S_pad - 1)];
  int all = 0, heads = 0, before = 0, mine = 0;      // of all tiles, of the heads before, of the head's tiles before the block's, of the head
  for (int base = 0; base < all_tiles; base += 256 * PER) {
    int w[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) w[k] = A.tile_bytes[min(base + 256 * k + tid, all_tiles - 1)];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int i = base + 256 * k + tid, x = i < all_tiles ? w[k] : 0;
      all += x; heads += i < head0 ? x : 0; before += i >= head0 && i < own0 ? x : 0; mine += i >= head0 && i < head0 + ntiles ? x : 0;
    }
  }
  u64 s0 = (u64)(u32)all | ((u64)(u32)heads << 32), s1 = (u64)(u32)before | ((u64)(u32)mine << 32);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) { s0 += __shfl_xor(s0, o, 64); s1 += __shfl_xor(s1, o, 64); }
  if (lane == 0) part[wave] = u32x4{(u32)s0, (u32)(s0 >> 32), (u32)s1, (u32)(s1 >> 32)};
  __syncthreads();
  const u32x4 sums = (part[0] + part[1]) + (part[2] + part[3]);
  all = (int)sums[0]; heads = (int)sums[1]; before = (int)sums[2]; mine = (int)sums[3];
  const bool fits = (long)all + 8 <= A.ovf_cap;
  if (blockIdx.x == 0 && tid == 0) {
    if (A.host_bytes) store_to_host(A.host_bytes + h, mine);
    A.head_bytes[h] = mine; A.head_start[h] = heads;
    if (h == H - 1) A.head_start[H] = all;
  }
  if (fits && blockIdx.x == 0 && h == H - 1 && tid < 8) A.ovf[all + tid] = 0;      // readers fetch eight bytes at a time
  // lane: a tile of the block
  n = tile0 + lane < ntiles ? n : 0;
  const int x = (int)row_scan16((u32)n), r0 = __builtin_amdgcn_readlane(x, 15), r1 = __builtin_amdgcn_readlane(x, 31), r2 = __builtin_amdgcn_readlane(x, 47);
  const int of = before + x + (lane >= 16 ? r0 : 0) + (lane >= 32 ? r1 : 0) + (lane >= 48 ? r2 : 0) - n;
  if (wave == 0 && tile0 + lane < ntiles) A.tile_off[head0 + tile0 + lane] = of;
#pragma unroll
  for (int k = 0; k < 4; ++k) {      // row offsets: tile offset + the escape bytes of the tile's earlier tag words
    const int i = t0 * T + 64 * k + lane;
    const u32 rb = (u32)esc_bytes(fl[k]), incl = row_scan16(rb);
    const int to = __shfl(of, 16 * wave + 4 * k + (lane >> 4), 64);
    if (i < A.S && n_own > 0) A.ovf_off[(long)h * A.S + i] = to + (int)(incl - rb);
  }
  if (!fits) return;
  uint8_t* dst = A.ovf + heads;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int nk = __builtin_amdgcn_readlane(n, 16 * wave + k), o = __builtin_amdgcn_readlane(of, 16 * wave + k);
    if (k >= n_own) break;
    if (lane < nk) dst[o + lane] = (uint8_t)v[k];
    for (int i = 64 + lane; i < nk; i += 64) dst[o + i] = src[esc_rest(t0 + k, ntiles) + i];
  }
}

// Two passes over the tag words of a head: escape bytes per chunk of 2048 rows, then per chunk the bytes of all earlier chunks (a
// short sum) plus a scan inside the chunk: 8 words per thread serially, thread totals by a block scan.
constexpr int RO_CHUNK = 2048;
__global__ void __launch_bounds__(256) k_row_chunk_sums(const int* __restrict__ flags, int S, int S_pad, int* __restrict__ chunk_sums) {
  __shared__ int sh[4];
  const int h = blockIdx.y, c = blockIdx.x, tid = threadIdx.x;
  const int* f = flags + (long)h * S_pad;
  const int s0 = c * RO_CHUNK + tid * 8;
  int mine = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) mine += s0 + k < S ? esc_bytes((u32)f[s0 + k]) : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mine += __shfl_xor(mine, o, 64);
  if ((tid & 63) == 0) sh[tid >> 6] = mine;
  __syncthreads();
  if (tid == 0) chunk_sums[(long)h * gridDim.x + c] = sh[0] + sh[1] + sh[2] + sh[3];
}
__global__ void __launch_bounds__(256) k_row_offsets(const int* __restrict__ flags, int S, int S_pad, const int* __restrict__ chunk_sums,
                                                     int* __restrict__ out) {
  __shared__ int sh[256];
  const int h = blockIdx.y, c = blockIdx.x, tid = threadIdx.x;
  const int* f = flags + (long)h * S_pad;
  int before = 0;
  for (int i = tid; i < c; i += 256) before += chunk_sums[(long)h * gridDim.x + i];
  const int s0 = c * RO_CHUNK + tid * 8;
  int rb[8], mine = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) { rb[k] = s0 + k < S ? esc_bytes((u32)f[s0 + k]) : 0; mine += rb[k]; }
  // block-wide: sum of `before`, inclusive scan of `mine`
  sh[tid] = before;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) { if (tid < o) sh[tid] += sh[tid + o]; __syncthreads(); }
  const int base = sh[0];
  __syncthreads();
  sh[tid] = mine;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    const int v = tid >= o ? sh[tid - o] : 0;
    __syncthreads();
    sh[tid] += v;
    __syncthreads();
  }
  int off = base + sh[tid] - mine;
#pragma unroll
  for (int k = 0; k < 8; ++k) { if (s0 + k < S) out[(long)h * S + s0 + k] = off; off += rb[k]; }
}

// ---------------------------------------------------------------------------------------------------- page decoder
// One wave per tile: short-lived waves at full occupancy overlap the dependent loads of a tile (tag words -> escape bytes) with the
// arithmetic and the stores of others (four tiles in a row per wave were a third slower; four waves a block: 8 x 65536 tokens 40.8 -> 41.6 us).
// Bound by the copy rate: 229 MB of a 64K-token page of 8 heads in 40.8 us = 5.6 TB/s in + out.  Before (bases read byte by byte from global
// memory, escape bytes one load after the other, rows stored through the caches) K took 47.6 and V 49.1; 8 x 16384: 13.6 and 15.4 -> 11.6.
struct DecodeArgs {
  const uint8_t* sm; const uint8_t* cd; const int* flags; const int* tile_off; const uint8_t* ovf; const int* head_start;
  const uint8_t* base3; const uint8_t* base4; int n_kv; const int* bidx; int S, S_pad; u16* out; long out_head_stride, out_row_stride;
};
template <int KIND>
__global__ void __launch_bounds__(64) k_decode_tiles(const DecodeArgs A) {
  __shared__ DecodeLds<KIND> L;
  const int lane = threadIdx.x, tile = blockIdx.x, h = blockIdx.y;
  const int brow = A.bidx ? A.bidx[h] : h % A.n_kv, nvalid = min(T, A.S - tile * T);
  const long row0 = (long)h * A.S_pad + (long)tile * T, boff = (long)brow * D;
  // rows beyond S carry tag 0 (the encoder writes every word of a tile) and are not written
  u16* dst = A.out + (long)h * A.out_head_stride + (long)tile * T * A.out_row_stride;
  const uint8_t* esc = A.ovf + A.head_start[h] + A.tile_off[(long)h * (A.S_pad / T) + tile];
  if ((A.out_row_stride & 7) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0)
    decode_tile_staged<KIND>(A.sm + row0 * D, A.cd + row0 * CB, A.flags + row0, esc, A.base3 + boff, A.base4 + boff, lane, nvalid, L, dst, A.out_row_stride);
  else      // rows that are not 16-byte aligned: element stores
    decode_tile_rows<KIND>(A.sm + row0 * D, A.cd + row0 * CB, A.flags + row0, esc, A.base3 + boff, A.base4 + boff, lane, nvalid, dst, A.out_row_stride);
}

// ---------------------------------------------------------------------------------------------------- prompt into the slot cache
// Per head, K and V: tile offsets and escape totals of the encoded tiles, the last L % 16 rows into the raw tail, and the head's counters.
// A head whose escapes do not fit its window (of K or of V) is left empty: the caller sees the totals, makes the windows larger and
// repeats the call.  One block per head.
struct PromptKind { const u16* x; long head_stride, row_stride; const int* tile_bytes; int* tile_off; u16* tail; int* ovf_used; };
struct PromptScanArgs { PromptKind j[2]; int n_kv, L, ntiles, off_stride, window; int* S; int* tail_len; int* head_bytes; };
__device__ __forceinline__ void copy_prompt_tail(const PromptScanArgs& A, const PromptKind& J, int h, int tid) {      // tid: 240 threads or more
  const int full = A.ntiles * T, row = tid >> 4, c16 = tid & 15;
  if (row < A.L - full)
    *reinterpret_cast<u32x4*>(J.tail + ((long)h * T + row) * D + 8 * c16) =
        *reinterpret_cast<const u32x4*>(J.x + (long)h * J.head_stride + (long)(full + row) * J.row_stride + 8 * c16);
}
__device__ __forceinline__ void set_prompt_counters(const PromptScanArgs& A, int kind, int h, int total, int other) {
  const PromptKind& J = A.j[kind];
  A.head_bytes[kind * A.n_kv + h] = total;
  const bool fits = A.ntiles == 0 || max(total, other) <= A.window;
  J.ovf_used[h] = fits ? total : 0;
  if (kind == 0) { A.S[h] = fits ? A.ntiles * T : 0; A.tail_len[h] = fits ? A.L - A.ntiles * T : 0; }
}
__global__ void __launch_bounds__(2 * SCAN_NT) k_prompt_scan(const PromptScanArgs A) {
  __shared__ int sh[2][SCAN_NT / 64];
  __shared__ int total[2];
  const int h = blockIdx.x, kind = threadIdx.x / SCAN_NT, tid = threadIdx.x % SCAN_NT;
  const PromptKind& J = A.j[kind];
  copy_prompt_tail(A, J, h, tid);
  const int mine = scan_tile_bytes(J.tile_bytes + (long)h * A.ntiles, J.tile_off + (long)h * A.off_stride, A.ntiles, tid, sh[kind]);
  if (tid == 0) total[kind] = mine;
  __syncthreads();
  if (tid == 0) set_prompt_counters(A, kind, h, mine, total[1 - kind]);
}
// The same and the packing (k_pack) in one launch, for prompts of up to PROMPT_PACK_TILES tiles: a block of 64 tiles adds up the sizes of all the
// head's tiles, and of those before its own, by itself (up to sixteen loads a thread in flight, from the L2) instead of waiting for a launch that
// does it.  Latency, like the two: 32768 tokens x 8 kv heads 8.9 us in two
// launches -> 4.8, 777 tokens 8.2 -> 5.3; the prompt of 32768 tokens 97.3 us a call -> 94.1.  Beyond, the blocks' reading of all sizes grows with the square of the length and k_prompt_scan + k_pack take over.
constexpr int PROMPT_PACK_TILES = 4096;
struct PromptPackArgs { PromptScanArgs s; const uint8_t* slots[2]; const int* head_start; uint8_t* ovf[2]; };
__global__ void __launch_bounds__(256) k_prompt_pack(const PromptPackArgs P) {
  __shared__ u64 part[4];
  __shared__ int part_other[4];
  const PromptScanArgs& A = P.s;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.y, kind = blockIdx.z, tile0 = blockIdx.x * PACK_TPB, ntiles = A.ntiles;
  const PromptKind& J = A.j[kind];
  const bool first = blockIdx.x == 0;
  if (ntiles == 0) {
    copy_prompt_tail(A, J, h, tid);
    if (tid == 0) set_prompt_counters(A, kind, h, 0, 0);
    return;
  }
  // every load up front, none under a branch; lane 16 r + c of the block takes piece c of the tail's row r
  const int tail_row = ntiles * T + (tid >> 4), head_start = P.head_start[h];
  const u32x4 tail = *reinterpret_cast<const u32x4*>(J.x + (long)h * J.head_stride + (long)min(tail_row, A.L - 1) * J.row_stride + 8 * (tid & 15));
  const int* tb = J.tile_bytes + (long)h * ntiles;
  const int* other = (first ? A.j[1 - kind].tile_bytes + (long)h * ntiles : tb);      // (only the first block needs them: no load under a branch)
  const uint8_t* src = P.slots[kind] + (long)h * ntiles * TILE_MAX_ESC;
  const int t0 = tile0 + 16 * wave, n_own = min(16, ntiles - t0);      // (may be <= 0)
  int n = tb[min(tile0 + lane, ntiles - 1)];
  u32 v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = src[(long)min(t0 + k, ntiles - 1) * ESC_HEAD + lane];
  int before = 0, all = 0, all_other = 0;
  for (int base = 0; base < ntiles; base += 256 * 8) {
    int w[8], x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) { const int i = min(base + 256 * k + tid, ntiles - 1); w[k] = tb[i]; x[k] = other[i]; }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = base + 256 * k + tid;
      all += i < ntiles ? w[k] : 0; before += i < tile0 ? w[k] : 0; all_other += i < ntiles ? x[k] : 0;
    }
  }
  u64 sums = (u64)(u32)all | ((u64)(u32)before << 32);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) { sums += __shfl_xor(sums, o, 64); all_other += __shfl_xor(all_other, o, 64); }
  if (lane == 0) { part[wave] = sums; part_other[wave] = all_other; }
  __syncthreads();
  sums = (part[0] + part[1]) + (part[2] + part[3]);
  all = (int)(u32)sums; before = (int)(sums >> 32);
  if (first && tid == 0) set_prompt_counters(A, kind, h, all, part_other[0] + part_other[1] + part_other[2] + part_other[3]);
  // lane: a tile of the block
  n = tile0 + lane < ntiles ? n : 0;
  const int x = (int)row_scan16((u32)n), r0 = __builtin_amdgcn_readlane(x, 15), r1 = __builtin_amdgcn_readlane(x, 31), r2 = __builtin_amdgcn_readlane(x, 47);
  const int of = before + x + (lane >= 16 ? r0 : 0) + (lane >= 32 ? r1 : 0) + (lane >= 48 ? r2 : 0) - n;
  if (wave == 0 && tile0 + lane < ntiles) J.tile_off[(long)h * A.off_stride + tile0 + lane] = of;
  if (first && tail_row < A.L) *reinterpret_cast<u32x4*>(J.tail + (long)h * T * D + 8 * tid) = tail;
  if (all > A.window) return;
  uint8_t* dst = P.ovf[kind] + head_start;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int nk = __builtin_amdgcn_readlane(n, 16 * wave + k), o = __builtin_amdgcn_readlane(of, 16 * wave + k);
    if (k >= n_own) break;
    if (lane < nk) dst[o + lane] = (uint8_t)v[k];
    for (int i = 64 + lane; i < nk; i += 64) dst[o + i] = src[esc_rest(t0 + k, ntiles) + i];
  }
}
// Short prompts (SCAN_PROMPT_TILES, SCAN_PROMPT_ALL_TILES): encoding, tile offsets and the escapes' way into the stream in one launch.  A block of four tiles says how many bytes it has
// in a 64-bit word that carries the launch's epoch, waits for the words of the head's earlier blocks and puts its escapes, which are in LDS until then, behind theirs.
// scan: words for K or V of a cache head, one and one for each of its blocks, zeroed once: the low half of [0] is the epoch of the last launch, which every block reads at its
// start and the head's last block, when it has seen the words of all, advances.  Launches on one cache head are ordered on a stream, as its contents demand.  A block
// waits for blocks with a smaller index, which start before it and wait only for smaller ones; the wait is bounded all the same.  A block that gives up, any of the
// head's, says so in the high half of [0] (its own size is out by then, so that the last block may see the words of all): k_prompt_finish, behind all blocks, then
// reports a negative total, which leaves the host's word unwritten (gaac_wait_words raises), and zeroes the words, some of which late blocks may have written.
// Latency: a launch less (5 us), against waiting for the slowest block ahead (2 to 3).  us a call, encoding and packing in two launches / in one: 300 tokens x 8 heads 18.5 /
// 15.9, 777 18.9 / 16.4, 777 x 16 19.6 / 17.4, 1500 x 8 (1488 tiles) 19.5 / 17.4, 2500 x 8 (2496) 20.1 / 19.1, 4095 x 2 (1020) 18.8 / 17.4; but 4095 x 8 (4080) 21.6 / 22.0: a
// chip full of blocks that wait.  (A block of sixteen waves for all tiles of a head, which has nobody to wait for: 777 tokens the same as two launches, 2047 30 us
// against 16.)
constexpr int SCAN_PROMPT_TILES = 256, SCAN_PROMPT_ALL_TILES = 3072, SCAN_SPIN_LIMIT = 1 << 20;      // of a head | of all heads, K and V
struct ScanWords { u64* k; long v; int row, spins; };      // K's of the call's first head, V's v words further on, row words a head (1 + blocks, or more); re-reads before a block gives up
struct PromptFusedArgs { EncodeArgs e; PromptScanArgs s; const int* head_start; uint8_t* ovf[2]; ScanWords scan; };
template <int KIND>
__device__ __forceinline__ void prompt_fused_body(const PromptFusedArgs& P, EncodeBlockLds& L, int (&sizes)[CODEC_WAVES], int& ahead, int h, int wave, int lane) {
  const EncodeArgs& A = P.e;
  const EncodeKind& J = KIND == KIND_K ? A.k : A.v;
  const PromptKind& K = P.s.j[KIND];
  const int ntiles = A.ntiles, block = blockIdx.x, tile = block * CODEC_WAVES + wave, brow = (A.brow0 + h) % A.NB;
  const int spins = P.scan.spins;
  asm volatile("" ::"s"(spins));      // with the other arguments: fetched where it is first used, behind the encoder, it made the launch 0.45 us longer
  u64* scan = P.scan.k + (KIND == KIND_V ? P.scan.v : 0) + (long)h * P.scan.row;
  const u16* xh = J.x + (long)h * J.head_stride;
  RowRegs R;
  load_rows<false>(R, xh + (long)min(tile, ntiles - 1) * T * J.row_stride, J.row_stride, T, lane);
  if (wave == 0) reinterpret_cast<u32x2*>(&L.B.w[0][0])[lane] = load_base_pair<KIND>(J.b3 + (long)brow * D, J.b4 + (long)brow * D, lane);
  u32* state = reinterpret_cast<u32*>(scan);      // epoch | whether a block gave up
  const u32 loaded_epoch = __hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int loaded_start = P.head_start[h];
  store_rows(L.w[wave], R, lane);
  // (waited for with the rows: where they are used the wait would be for the encoder's stores as well)
  const u32 last = (u32)__builtin_amdgcn_readfirstlane((int)loaded_epoch), epoch = last + (last == 0xFFFFFFFFu ? 2u : 1u);      // (0 is what the words start with)
  const int head_start = __builtin_amdgcn_readfirstlane(loaded_start);
  __syncthreads();
  int total = 0;
  const uint8_t* escapes = nullptr;
  if (tile < ntiles) {
    const long row0 = (long)h * A.S_pad + (long)tile * T;
    UnitEscapes E;
    total = encode_staged_tile<KIND, true>(L.w[wave], L.B, T, lane, J.sm + row0 * D, J.cd + row0 * CB, J.flags + row0, E);
    escapes = collect_escapes<KIND>(L.w[wave], E, lane);
  }
  if (lane == 0) sizes[wave] = total;
  __syncthreads();
  const int own = sizes[0] + sizes[1] + sizes[2] + sizes[3];
  if (wave == 0) {
    if (lane == 0) __hip_atomic_store(scan + 1 + block, (u64)(u32)own | ((u64)epoch << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // lane: an earlier block (64 blocks at most; the others read the block's own word)
    const u64* w = scan + 1 + min(lane, block);
    u64 v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool ok = true;
    for (int spin = 0; __builtin_amdgcn_ballot_w64(lane < block && (u32)(v >> 32) != epoch) != 0; ++spin) {
      if (spin >= spins) { ok = false; break; }
      __builtin_amdgcn_s_sleep(1);
      if ((u32)(v >> 32) != epoch) v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int x = (int)row_scan16(lane < block ? (u32)v : 0u);
    const int before = __builtin_amdgcn_readlane(x, 15) + __builtin_amdgcn_readlane(x, 31) + __builtin_amdgcn_readlane(x, 47) + __builtin_amdgcn_readlane(x, 63);
    if (lane == 0) {
      ahead = ok ? before : -1;
      if (!ok) __hip_atomic_store(state + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else if (block == (ntiles - 1) / CODEC_WAVES) {
        P.s.head_bytes[KIND * P.s.n_kv + h] = before + own;
        __hip_atomic_store(state, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (block == 0) copy_prompt_tail(P.s, K, h, 64 * wave + lane);
  __syncthreads();
  int at = ahead;
  if (at < 0 || tile >= ntiles) return;
#pragma unroll
  for (int w = 0; w < CODEC_WAVES; ++w) at += w < wave ? sizes[w] : 0;
  if (lane == 0) K.tile_off[(long)h * P.s.off_stride + tile] = at;
  if (at + total > P.s.window) return;      // (the head does not fit and is left empty)
  uint8_t* dst = P.ovf[KIND] + head_start + at;
  for (int i = lane; i < total; i += 64) dst[i] = escapes[i];
}
__global__ void __launch_bounds__(64 * CODEC_WAVES) k_prompt_fused(const PromptFusedArgs P) {
  __shared__ EncodeBlockLds L;
  __shared__ int sizes[CODEC_WAVES], ahead;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (blockIdx.z == KIND_K) prompt_fused_body<KIND_K>(P, L, sizes, ahead, blockIdx.y, wave, lane);
  else prompt_fused_body<KIND_V>(P, L, sizes, ahead, blockIdx.y, wave, lane);
}
// ... and the counters of the heads, with the totals in host memory as k_words_to_host puts them there.
__global__ void __launch_bounds__(64) k_prompt_finish(const PromptScanArgs A, const ScanWords W, int* __restrict__ host) {
  for (int h = threadIdx.x; h < A.n_kv; h += 64) {
    u64 *kw = W.k + (long)h * W.row, *vw = kw + W.v;
    // (one trip to memory for all four; the rest is as if none had given up, where none has)
    const u32 k_gave_up = reinterpret_cast<const u32*>(kw)[1], v_gave_up = reinterpret_cast<const u32*>(vw)[1];
    int k = A.head_bytes[h], v = A.head_bytes[A.n_kv + h];
    const bool failed = (k_gave_up | v_gave_up) != 0u;
    k = k_gave_up ? -1 : k; v = v_gave_up ? -1 : v;
    const int least = failed ? 0x7FFFFFFF : 0;      // (a total that fits no window)
    set_prompt_counters(A, KIND_K, h, max(k, least), max(v, least));
    set_prompt_counters(A, KIND_V, h, max(v, least), max(k, least));
    if (failed) {      // all blocks are through: the words start anew (all of them: the epoch is 1 next, which an old launch may have left)
      A.head_bytes[h] = k; A.head_bytes[A.n_kv + h] = v;
      for (int i = 0; i < W.row; ++i) { if (k_gave_up) kw[i] = 0ull; if (v_gave_up) vw[i] = 0ull; }
    }
    if (host) { store_to_host(host + h, k); store_to_host(host + A.n_kv + h, v); }
  }
}
// The prompt's totals into host memory that the host polls, in a launch of its own: by the time they are there all of the prompt is.  Polling spares
// the host the 5 us that a stream's synchronisation takes from the end of its last kernel, for 2 of this launch: a prompt of 777 tokens 26 -> 21.5 us a call,
// of 32768 95.8 -> 91.4, the case of four short requests 363 -> 308.
__global__ void __launch_bounds__(64) k_words_to_host(const int* __restrict__ words, int n, int* __restrict__ host) {
  for (int i = threadIdx.x; i < n; i += 64) store_to_host(host + i, words[i]);
}

}  // namespace gaac

using namespace gaac;

extern "C" {

const char* gaac_last_error(void) { return last_error_buffer(); }

int gaac_wait_words(const int* words, int n, void* stream) {
  GAAC_REQUIRE(words && n > 0, "gaac_wait_words: bad arguments");
  const auto there = [&] {
    for (int i = 0; i < n; ++i) if (__atomic_load_n(words + i, __ATOMIC_ACQUIRE) < 0) return false;
    return true;
  };
  const auto give_up = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
  do {
    for (int spin = 0; spin < 64; ++spin) if (there()) return 0;
  } while (std::chrono::steady_clock::now() < give_up);
  const hipError_t e = hipStreamSynchronize((hipStream_t)stream);      // a busy stream, or one that failed
  if (e != hipSuccess) return gaac::fail("gaac_wait_words: %s", hipGetErrorString(e));
  GAAC_REQUIRE(there(), "gaac_wait_words: the stream is done and has not written all words");
  return 0;
}

int gaac_exponent_hist(const void* x, long n_tokens, int n_kv, long long* hist, void* stream) {
  GAAC_REQUIRE(x && hist && n_kv > 0 && n_tokens >= 0, "gaac_exponent_hist: bad arguments");
  if (n_tokens == 0) return 0;
  const long row = (long)n_kv * D;
  HistArgs A{{(const u16*)x, nullptr}, {D, 0}, {row, 0}, n_tokens, 0, n_kv, (unsigned long long*)hist, nullptr, nullptr};
  launch_hist(A, 1, hist_chunks(n_tokens, n_kv, false), (hipStream_t)stream);
  return launch_status("gaac_exponent_hist");
}

int gaac_bases_from_hist(const long long* hist, int rows, uint8_t* base3, uint8_t* base4, void* stream) {
  GAAC_REQUIRE(hist && base3 && base4 && rows > 0, "gaac_bases_from_hist: bad arguments");
  hipLaunchKernelGGL(k_bases_from_hist, dim3((rows + 3) / 4), dim3(256), 0, (hipStream_t)stream, hist, rows, base3, base4);
  return launch_status("gaac_bases_from_hist");
}

int gaac_encode_tiles(int kind, const void* x, long x_head_stride, long x_row_stride, int H, int S, int S_pad, const uint8_t* base3,
                      const uint8_t* base4, int n_kv, const int* bidx, uint8_t* sm, uint8_t* codes, int* flags, uint8_t* esc_slots,
                      int* tile_bytes, void* stream) {
  GAAC_REQUIRE(kind == 0 || kind == 1, "gaac_encode_tiles: kind must be 0 (k) or 1 (v)");
  GAAC_REQUIRE(x && base3 && base4 && sm && codes && flags && esc_slots && tile_bytes, "gaac_encode_tiles: null pointer");
  GAAC_REQUIRE(H > 0 && S > 0 && S_pad >= (S + T - 1) / T * T && S_pad % T == 0 && n_kv > 0,
               "gaac_encode_tiles: bad sizes H=%d S=%d S_pad=%d n_kv=%d", H, S, S_pad, n_kv);
  GAAC_REQUIRE(x_row_stride >= D && x_row_stride % 8 == 0 && x_head_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0,
               "gaac_encode_tiles: rows must be 16-byte aligned (strides in elements: head %ld, row %ld)", x_head_stride, x_row_stride);
  EncodeArgs A{};
  A.kind0 = kind; A.S = S; A.S_pad = S_pad; A.ntiles = (S + T - 1) / T; A.brow0 = 0; A.NB = n_kv; A.bidx = bidx;
  (kind == 0 ? A.k : A.v) = EncodeKind{(const u16*)x, x_head_stride, x_row_stride, base3, base4, sm, codes, flags, esc_slots, tile_bytes};
  launch_encode<false>(A, H, 1, (hipStream_t)stream);
  return launch_status("gaac_encode_tiles");
}

int gaac_tile_scan(const int* tile_bytes, int H, int ntiles, int* tile_off, int* head_bytes, int* host_bytes, void* stream) {
  GAAC_REQUIRE(tile_bytes && tile_off && head_bytes && H > 0 && ntiles > 0, "gaac_tile_scan: bad arguments");
  hipLaunchKernelGGL(k_tile_scan, dim3(H), dim3(SCAN_NT), 0, (hipStream_t)stream, tile_bytes, tile_off, ntiles, head_bytes, host_bytes);
  return launch_status("gaac_tile_scan");
}

int gaac_page_pack(const uint8_t* esc_slots, const int* tile_bytes, const int* tile_off, const int* head_bytes, const int* flags, int H, int S, int S_pad,
                   int* head_start, uint8_t* ovf, int* ovf_off, void* stream) {
  GAAC_REQUIRE(esc_slots && tile_bytes && tile_off && head_bytes && flags && head_start && ovf && ovf_off, "gaac_page_pack: null pointer");
  GAAC_REQUIRE(H > 0 && S > 0 && S_pad >= (S + T - 1) / T * T && S_pad % T == 0, "gaac_page_pack: bad sizes H=%d S=%d S_pad=%d", H, S, S_pad);
  PackArgs A{};
  A.ntiles = (S + T - 1) / T;
  A.j[0] = PackKind{esc_slots, tile_bytes, tile_off, A.ntiles, nullptr, ovf};
  A.head_bytes = head_bytes; A.flags = flags; A.S = S; A.S_pad = S_pad; A.head_start_out = head_start; A.ovf_off = ovf_off; A.ovf_cap = 0x7FFFFFFFL + 8;
  hipLaunchKernelGGL(k_pack<true>, dim3((A.ntiles + PACK_TPB - 1) / PACK_TPB, H), dim3(256), 0, (hipStream_t)stream, A);
  return launch_status("gaac_page_pack");
}

int gaac_page_finish(const uint8_t* esc_slots, const int* tile_bytes, const int* flags, int H, int S, int S_pad, int* tile_off, int* head_bytes,
                     int* host_bytes, int* head_start, uint8_t* ovf, long ovf_cap, int* ovf_off, void* stream) {
  GAAC_REQUIRE(esc_slots && tile_bytes && tile_off && head_bytes && host_bytes && flags && head_start && ovf && ovf_off, "gaac_page_finish: null pointer");
  GAAC_REQUIRE(H > 0 && S > 0 && S_pad >= (S + T - 1) / T * T && S_pad % T == 0 && ovf_cap >= 8, "gaac_page_finish: bad sizes H=%d S=%d S_pad=%d ovf_cap=%ld", H, S, S_pad, ovf_cap);
  hipStream_t st = (hipStream_t)stream;
  const int ntiles = (S + T - 1) / T;
  const dim3 grid((ntiles + PACK_TPB - 1) / PACK_TPB, H);
  for (int h = 0; h < H; ++h) __atomic_store_n(host_bytes + h, -1, __ATOMIC_RELAXED);      // not there yet
  if ((long)H * ntiles <= PAGE_PACK_TILES) {
    const PagePackArgs A{esc_slots, tile_bytes, tile_off, head_bytes, host_bytes, ntiles, flags, S, S_pad, head_start, ovf, ovf_cap, ovf_off};
    hipLaunchKernelGGL(k_page_pack, grid, dim3(256), 0, st, A);
  } else {
    hipLaunchKernelGGL(k_tile_scan, dim3(H), dim3(SCAN_NT), 0, st, tile_bytes, tile_off, ntiles, head_bytes, host_bytes);
    PackArgs A{};
    A.ntiles = ntiles;
    A.j[0] = PackKind{esc_slots, tile_bytes, tile_off, ntiles, nullptr, ovf};
    A.head_bytes = head_bytes; A.flags = flags; A.S = S; A.S_pad = S_pad; A.head_start_out = head_start; A.ovf_off = ovf_off; A.ovf_cap = ovf_cap;
    hipLaunchKernelGGL(k_pack<true>, grid, dim3(256), 0, st, A);
  }
  return launch_status("gaac_page_finish");
}

int gaac_compact(const uint8_t* esc_slots, const int* tile_bytes, int* tile_off, const int* head_start, uint8_t* ovf,
                 int H, int ntiles, void* stream) {
  GAAC_REQUIRE(esc_slots && tile_bytes && tile_off && head_start && ovf && H > 0 && ntiles > 0, "gaac_compact: bad arguments");
  hipLaunchKernelGGL(k_tile_scan, dim3(H), dim3(SCAN_NT), 0, (hipStream_t)stream, tile_bytes, tile_off, ntiles, (int*)nullptr, (int*)nullptr);
  PackArgs A{};
  A.ntiles = ntiles;
  A.j[0] = PackKind{esc_slots, tile_bytes, tile_off, ntiles, head_start, ovf};
  hipLaunchKernelGGL(k_pack<false>, dim3((ntiles + PACK_TPB - 1) / PACK_TPB, H), dim3(256), 0, (hipStream_t)stream, A);
  return launch_status("gaac_compact");
}

int gaac_row_offsets(const int* flags, int H, int S, int S_pad, int* chunk_sums, int* out, void* stream) {
  GAAC_REQUIRE(flags && out && chunk_sums && H > 0 && S > 0 && S_pad >= S, "gaac_row_offsets: bad arguments");
  const dim3 grid((S + RO_CHUNK - 1) / RO_CHUNK, H);
  hipLaunchKernelGGL(k_row_chunk_sums, grid, dim3(256), 0, (hipStream_t)stream, flags, S, S_pad, chunk_sums);
  hipLaunchKernelGGL(k_row_offsets, grid, dim3(256), 0, (hipStream_t)stream, flags, S, S_pad, chunk_sums, out);
  return launch_status("gaac_row_offsets");
}

int gaac_decode_tiles(int kind, const uint8_t* sm, const uint8_t* codes, const int* flags, const int* tile_off, const uint8_t* ovf,
                      const int* head_start, const uint8_t* base3, const uint8_t* base4, int n_kv, const int* bidx, int H, int S,
                      int S_pad, void* out, long out_head_stride, long out_row_stride, void* stream) {
  GAAC_REQUIRE(kind == 0 || kind == 1, "gaac_decode_tiles: kind must be 0 (k) or 1 (v)");
  GAAC_REQUIRE(sm && codes && flags && tile_off && ovf && head_start && base3 && base4 && out, "gaac_decode_tiles: null pointer");
  GAAC_REQUIRE(H > 0 && S > 0 && S_pad >= (S + T - 1) / T * T && S_pad % T == 0 && n_kv > 0, "gaac_decode_tiles: bad sizes");
  const DecodeArgs A{sm, codes, flags, tile_off, ovf, head_start, base3, base4, n_kv, bidx, S, S_pad, (u16*)out, out_head_stride, out_row_stride};
  const dim3 grid((S + T - 1) / T, H);
  if (kind == 0) hipLaunchKernelGGL(k_decode_tiles<KIND_K>, grid, dim3(64), 0, (hipStream_t)stream, A);
  else hipLaunchKernelGGL(k_decode_tiles<KIND_V>, grid, dim3(64), 0, (hipStream_t)stream, A);
  return launch_status("gaac_decode_tiles");
}

// hist_bytes < 0: hist as gaac_cache_prefill takes it, 2^17 bytes for K and for V of each head, which are a table; prompts that want more tables, or need
// them, have them where their escapes will be (1280 bytes a tile against a table for 256 tokens or more).
static int prompt_store(
    const char* name,
    const void* k, const void* v, long k_head_stride, long k_row_stride, long v_head_stride, long v_row_stride, int L, int n_kv, int head0,
    int cap, int ovf_cap, int NB, int calibrate, int* tail_len, int* S, const int* head_start,
    void* k_tail, uint8_t* k_base3, uint8_t* k_base4, uint8_t* k_sm, uint8_t* k_codes, int* k_flags, uint8_t* k_ovf, int* k_tile_off, int* k_ovf_used,
    void* v_tail, uint8_t* v_base3, uint8_t* v_base4, uint8_t* v_sm, uint8_t* v_codes, int* v_flags, uint8_t* v_ovf, int* v_tile_off, int* v_ovf_used,
    void* hist, long hist_bytes, uint8_t* esc_slots, int* tile_bytes, int* head_bytes, const ScanWords& scan, int* host_bytes, void* stream) {
  GAAC_REQUIRE(((k && v) || L == 0) && tail_len && S && head_start && head_bytes, "%s: null pointer", name);
  GAAC_REQUIRE(k_tail && k_base3 && k_base4 && k_sm && k_codes && k_flags && k_ovf && k_tile_off && k_ovf_used, "%s: null K store pointer", name);
  GAAC_REQUIRE(v_tail && v_base3 && v_base4 && v_sm && v_codes && v_flags && v_ovf && v_tile_off && v_ovf_used, "%s: null V store pointer", name);
  GAAC_REQUIRE(L >= 0 && n_kv > 0 && head0 >= 0 && cap > 0 && cap % T == 0 && L <= cap && NB > 0 && ovf_cap >= 8,
               "%s: bad sizes L=%d n_kv=%d head0=%d cap=%d ovf_cap=%d NB=%d", name, L, n_kv, head0, cap, ovf_cap, NB);
  GAAC_REQUIRE(!calibrate || (hist && NB >= head0 + n_kv), "%s: calibration needs its scratch and a base row per cache head (NB=%d, heads %d..%d)", name, NB, head0, head0 + n_kv - 1);
  const int ntiles = L / T;
  GAAC_REQUIRE(ntiles == 0 || (esc_slots && tile_bytes), "%s: null scratch", name);
  GAAC_REQUIRE(L == 0 || (k_row_stride >= D && k_row_stride % 8 == 0 && k_head_stride % 8 == 0 && v_row_stride >= D && v_row_stride % 8 == 0 && v_head_stride % 8 == 0 &&
                          ((reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15) == 0), "%s: rows must be 16-byte aligned", name);
  int tables = calibrate ? hist_chunks(L, 2 * n_kv, true) : 0;      // of a (kind, head)
  if (calibrate && hist_bytes < 0) {
    const long room = (2l * n_kv * ntiles * TILE_MAX_ESC - 8) / (2 * n_kv * HIST_TABLE);
    if (room >= 2 && tables >= 2) { hist = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(esc_slots) + 7) & ~(uintptr_t)7); tables = (int)std::min<long>(tables, room); }
    else tables = 1;
  } else if (calibrate) GAAC_REQUIRE(2l * n_kv * tables * HIST_TABLE <= hist_bytes, "%s: %ld bytes of calibration scratch for %ld tables", name, hist_bytes, 2l * n_kv * tables);
  GAAC_REQUIRE(!calibrate || (reinterpret_cast<uintptr_t>(hist) & 7) == 0, "%s: calibration scratch is not aligned to 8 bytes", name);
  hipStream_t st = (hipStream_t)stream;
  if (calibrate) {
    u32* rows = (u32*)hist;
    u16* bits = reinterpret_cast<u16*>(rows + 2l * n_kv * tables * (256 * 64));
    HistArgs H{{(const u16*)k, (const u16*)v}, {k_head_stride, v_head_stride}, {k_row_stride, v_row_stride}, L, 0, n_kv, nullptr, rows, bits};
    const int chunks = L > 0 ? launch_hist(H, 2, tables, st) : 0;
    const PromptBasesArgs B{rows, bits, chunks, {k_base3, v_base3}, {k_base4, v_base4}, n_kv, head0};
    // (as many loads in flight as there are tables for: a lane past the last table reads that one again)
    if (chunks <= 16) hipLaunchKernelGGL(k_prompt_bases<4>, dim3(4, n_kv, 2), dim3(1024), 0, st, B);
    else if (chunks <= 32) hipLaunchKernelGGL(k_prompt_bases<8>, dim3(4, n_kv, 2), dim3(1024), 0, st, B);
    else hipLaunchKernelGGL(k_prompt_bases<16>, dim3(4, n_kv, 2), dim3(1024), 0, st, B);
  }
  const long row0 = (long)head0 * cap, tile0 = (long)head0 * (cap / T), n_all = (long)n_kv * ntiles;
  uint8_t* v_slots = esc_slots ? esc_slots + n_all * TILE_MAX_ESC : nullptr;
  int* v_bytes = tile_bytes ? tile_bytes + n_all : nullptr;
  const int nblocks = (ntiles + CODEC_WAVES - 1) / CODEC_WAVES;
  const bool fused = scan.k && ntiles > 0 && ntiles <= SCAN_PROMPT_TILES && 2 * n_all <= SCAN_PROMPT_ALL_TILES && nblocks < scan.row;
  EncodeArgs E{};
  if (ntiles > 0) {
    E.kind0 = KIND_K; E.S = ntiles * T; E.S_pad = cap; E.ntiles = ntiles; E.brow0 = head0; E.NB = NB; E.bidx = nullptr;
    E.k = EncodeKind{(const u16*)k, k_head_stride, k_row_stride, k_base3, k_base4, k_sm + row0 * D, k_codes + row0 * CB, k_flags + row0, esc_slots, tile_bytes};
    E.v = EncodeKind{(const u16*)v, v_head_stride, v_row_stride, v_base3, v_base4, v_sm + row0 * D, v_codes + row0 * CB, v_flags + row0, v_slots, v_bytes};
    if (!fused) launch_encode<true>(E, n_kv, 2, st);
  }
  const int window = ovf_cap - (TILE_MAX_ESC + 8);      // room for one more worst-case tile and the readers' padding stays free
  PromptScanArgs P{};
  P.j[0] = PromptKind{(const u16*)k, k_head_stride, k_row_stride, tile_bytes, k_tile_off + tile0, (u16*)k_tail + (long)head0 * T * D, k_ovf_used + head0};
  P.j[1] = PromptKind{(const u16*)v, v_head_stride, v_row_stride, v_bytes, v_tile_off + tile0, (u16*)v_tail + (long)head0 * T * D, v_ovf_used + head0};
  P.n_kv = n_kv; P.L = L; P.ntiles = ntiles; P.off_stride = cap / T; P.window = window;
  P.S = S + head0; P.tail_len = tail_len + head0; P.head_bytes = head_bytes;
  if (host_bytes) for (int i = 0; i < 2 * n_kv; ++i) __atomic_store_n(host_bytes + i, -1, __ATOMIC_RELAXED);      // not there yet
  if (fused) {
    const PromptFusedArgs A{E, P, head_start + head0, {k_ovf, v_ovf}, scan};
    hipLaunchKernelGGL(k_prompt_fused, dim3(nblocks, n_kv, 2), dim3(64 * CODEC_WAVES), 0, st, A);
    hipLaunchKernelGGL(k_prompt_finish, dim3(1), dim3(64), 0, st, P, scan, host_bytes);
    return launch_status(name);
  }
  if (ntiles <= PROMPT_PACK_TILES) {
    const PromptPackArgs A{P, {esc_slots, v_slots}, head_start + head0, {k_ovf, v_ovf}};
    hipLaunchKernelGGL(k_prompt_pack, dim3(std::max((ntiles + PACK_TPB - 1) / PACK_TPB, 1), n_kv, 2), dim3(256), 0, st, A);
  } else {
    hipLaunchKernelGGL(k_prompt_scan, dim3(n_kv), dim3(2 * SCAN_NT), 0, st, P);
    PackArgs A{};
    A.ntiles = ntiles; A.head_bytes = head_bytes; A.window = window;
    A.j[0] = PackKind{esc_slots, tile_bytes, k_tile_off + tile0, cap / T, head_start + head0, k_ovf};
    A.j[1] = PackKind{v_slots, v_bytes, v_tile_off + tile0, cap / T, head_start + head0, v_ovf};
    hipLaunchKernelGGL(k_pack<false>, dim3((ntiles + PACK_TPB - 1) / PACK_TPB, n_kv, 2), dim3(256), 0, st, A);
  }
  if (host_bytes) hipLaunchKernelGGL(k_words_to_host, dim3(1), dim3(64), 0, st, head_bytes, 2 * n_kv, host_bytes);
  return launch_status(name);
}

int gaac_prompt_store(
    const void* k, const void* v, long k_head_stride, long k_row_stride, long v_head_stride, long v_row_stride, int L, int n_kv, int head0,
    int cap, int ovf_cap, int NB, int calibrate, int* tail_len, int* S, const int* head_start,
    void* k_tail, uint8_t* k_base3, uint8_t* k_base4, uint8_t* k_sm, uint8_t* k_codes, int* k_flags, uint8_t* k_ovf, int* k_tile_off, int* k_ovf_used,
    void* v_tail, uint8_t* v_base3, uint8_t* v_base4, uint8_t* v_sm, uint8_t* v_codes, int* v_flags, uint8_t* v_ovf, int* v_tile_off, int* v_ovf_used,
    void* hist, long hist_bytes, uint8_t* esc_slots, int* tile_bytes, int* head_bytes, unsigned long long* scan, long scan_v, int scan_row, int scan_spins,
    int* host_bytes, void* stream) {
  GAAC_REQUIRE(hist_bytes >= 0 && scan_spins >= 0 && (!scan || scan_row > 0), "gaac_prompt_store: bad sizes hist_bytes=%ld scan_row=%d scan_spins=%d", hist_bytes, scan_row, scan_spins);
  return prompt_store("gaac_prompt_store", k, v, k_head_stride, k_row_stride, v_head_stride, v_row_stride, L, n_kv, head0, cap, ovf_cap, NB, calibrate, tail_len, S, head_start,
                      k_tail, k_base3, k_base4, k_sm, k_codes, k_flags, k_ovf, k_tile_off, k_ovf_used, v_tail, v_base3, v_base4, v_sm, v_codes, v_flags, v_ovf, v_tile_off, v_ovf_used,
                      hist, hist_bytes, esc_slots, tile_bytes, head_bytes, ScanWords{reinterpret_cast<u64*>(scan), scan_v, scan_row, scan_spins ? scan_spins : SCAN_SPIN_LIMIT}, host_bytes, stream);
}

int gaac_cache_prefill(
    const void* k, const void* v, long k_head_stride, long k_row_stride, long v_head_stride, long v_row_stride, int L, int n_kv, int head0,
    int cap, int ovf_cap, int NB, int calibrate, int* tail_len, int* S, const int* head_start,
    void* k_tail, uint8_t* k_base3, uint8_t* k_base4, uint8_t* k_sm, uint8_t* k_codes, int* k_flags, uint8_t* k_ovf, int* k_tile_off, int* k_ovf_used,
    void* v_tail, uint8_t* v_base3, uint8_t* v_base4, uint8_t* v_sm, uint8_t* v_codes, int* v_flags, uint8_t* v_ovf, int* v_tile_off, int* v_ovf_used,
    unsigned long long* hist, uint8_t* esc_slots, int* tile_bytes, int* head_bytes, int* host_bytes, void* stream) {
  return prompt_store("gaac_cache_prefill", k, v, k_head_stride, k_row_stride, v_head_stride, v_row_stride, L, n_kv, head0, cap, ovf_cap, NB, calibrate, tail_len, S, head_start,
                      k_tail, k_base3, k_base4, k_sm, k_codes, k_flags, k_ovf, k_tile_off, k_ovf_used, v_tail, v_base3, v_base4, v_sm, v_codes, v_flags, v_ovf, v_tile_off, v_ovf_used,
                      hist, -1, esc_slots, tile_bytes, head_bytes, ScanWords{}, host_bytes, stream);
}

}  // extern "C"
