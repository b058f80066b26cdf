// Calibration, page encoder and page decoder kernels + their extern "C" entry points.
//   exponent_hist / bases_from_hist   /root/reference/gaac/codec.py:70-84
//   encode_tiles / compact            /root/reference/gaac/encoder.py:16-76, 94-109
//   row_offsets                       /root/reference/gaac/codec.py:221-225
//   decode_tiles                      /root/reference/gaac/codec.py:186-218
#include "gaac_tile.h"
#include "gaac_capi.h"
#include "../../include/gaac_hip.h"

namespace gaac {

char* last_error_buffer() { static thread_local char buf[512] = {0}; return buf; }

// ---------------------------------------------------------------------------------------------------- calibration
// Exponent histogram per (kv head, channel).  A block owns 64 channels of the n_kv*128-wide token row and a chunk of tokens: eight
// lanes read the 128 bytes of a row with 16-byte loads, counts go to LDS (64 x 256 x 4 B) and from there, where non-zero, to the
// 64-bit global histogram.
constexpr int HIST_CH = 64;
__global__ void __launch_bounds__(256) k_exponent_hist(const u16* __restrict__ x, long n_tok, int n_kv, int chunk,
                                                       unsigned long long* __restrict__ hist) {
  __shared__ u32 h[HIST_CH * 256];
  const int tid = threadIdx.x, c0 = blockIdx.x * HIST_CH;      // first of this block's channels in the n_kv*128 row
  for (int i = tid; i < HIST_CH * 256; i += 256) h[i] = 0u;
  __syncthreads();
  const long t0 = (long)blockIdx.y * chunk, t1 = min(t0 + (long)chunk, n_tok);
  const int c8 = tid & 7, sub = tid >> 3;
  const long row = (long)n_kv * D;
  const u16* xp = x + c0 + 8 * c8;
  u32* hc = h + (8 * c8) * 256;
  for (long t = t0 + sub; t < t1; t += 4 * 32) {      // four rows in flight per thread
    u32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = t + 32 * k < t1 ? *reinterpret_cast<const u32x4*>(xp + (t + 32 * k) * row) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (t + 32 * k >= t1) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        atomicAdd(&hc[(2 * j) * 256 + ((v[k][j] >> 7) & 0xFFu)], 1u);
        atomicAdd(&hc[(2 * j + 1) * 256 + ((v[k][j] >> 23) & 0xFFu)], 1u);
      }
    }
  }
  __syncthreads();
  for (int i = tid; i < HIST_CH * 256; i += 256)
    if (h[i]) atomicAdd(&hist[(long)(c0 + (i >> 8)) * 256 + (i & 255)], (unsigned long long)h[i]);
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
// A block of four waves takes 4 * TPW consecutive tiles of one head, wave w the tiles w, w+4, ... of them (one-wave blocks, one per tile,
// would be limited by the rate at which workgroups can be launched).  The rows of a wave's next tile are fetched into registers while it
// encodes the current one.  K and V of a prompt share a launch (blockIdx.z): one start-up and one drain for both.
constexpr int CODEC_WAVES = 4;
struct EncodeKind {      // one of K, V
  const u16* x; long head_stride, row_stride;
  const uint8_t* b3; const uint8_t* b4;
  uint8_t* sm; uint8_t* cd; int* flags;            // head 0 of the call; token stride S_pad
  uint8_t* slots; int* tile_bytes;                 // [H][ntiles] worst-case escape slots and the bytes used in each
};
struct EncodeArgs { EncodeKind k, v; int kind0, S, S_pad, ntiles, brow0, NB; const int* bidx; };      // blockIdx.z = 0 is kind0
template <int KIND, int TPW>
__device__ __forceinline__ void encode_tiles_body(const EncodeArgs& A, const EncodeKind& J, EncodeLds& L, int h, int tile, int lane) {
  const int S = A.S, ntiles = A.ntiles;
  const int brow = A.bidx ? A.bidx[h] : (A.brow0 + h) % A.NB;
  const u16* xh = J.x + (long)h * J.head_stride;
  RowRegs R, Rn;
  load_rows(R, xh + (long)tile * T * J.row_stride, J.row_stride, min(T, S - tile * T), lane);
  stage_bases(L, J.b3 + (long)brow * D, J.b4 + (long)brow * D, lane);
  wave_lds_sync();
  BaseRegs Bs;                // the base words of the lane's units: the same for every tile of the head
  load_base_regs<KIND>(L, lane & 15, lane >> 4, Bs);
  for (int i = 0; i < TPW && tile < ntiles; ++i, tile += CODEC_WAVES) {
    const int nvalid = min(T, S - tile * T), next = tile + CODEC_WAVES;
    store_rows(L, R, lane);
    if (i + 1 < TPW && next < ntiles) load_rows(Rn, xh + (long)next * T * J.row_stride, J.row_stride, min(T, S - next * T), lane);
    wave_lds_sync();
    const long row0 = (long)h * A.S_pad + (long)tile * T;
    const int total = encode_staged_tile<KIND>(L, Bs, nvalid, lane, J.sm + row0 * D, J.cd + row0 * CB, J.flags + row0,
                                               J.slots + ((long)h * ntiles + tile) * TILE_MAX_ESC);
    if (lane == 0) J.tile_bytes[(long)h * ntiles + tile] = total;
    wave_lds_sync();          // the staged rows and tag words are free again
    R = Rn;
  }
}
template <int TPW>
__global__ void __launch_bounds__(64 * CODEC_WAVES) k_encode_tiles(const EncodeArgs A) {
  __shared__ EncodeLds Ls[CODEC_WAVES];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, tile = blockIdx.x * (CODEC_WAVES * TPW) + wave;
  if (tile >= A.ntiles) return;
  if (A.kind0 + (int)blockIdx.z == KIND_K) encode_tiles_body<KIND_K, TPW>(A, A.k, Ls[wave], blockIdx.y, tile, lane);
  else encode_tiles_body<KIND_V, TPW>(A, A.v, Ls[wave], blockIdx.y, tile, lane);
}
static void launch_encode(const EncodeArgs& A, int H, int kinds, hipStream_t stream) {
  // Four tiles in a row per wave hide a tile's row loads behind the previous tile and share the base words; below 8192 tiles (eight
  // waves per SIMD with one tile each) that leaves SIMDs idle, and one tile per wave is faster:
  // 7.9 against 10.4 us at 2048 tiles, 17.8 against 15.8 us at 8192, 56 against 52 us at 32768
  if ((long)A.ntiles * H * kinds >= 8192)
    hipLaunchKernelGGL(k_encode_tiles<4>, dim3((A.ntiles + 4 * CODEC_WAVES - 1) / (4 * CODEC_WAVES), H, kinds), dim3(64 * CODEC_WAVES), 0, stream, A);
  else
    hipLaunchKernelGGL(k_encode_tiles<1>, dim3((A.ntiles + CODEC_WAVES - 1) / CODEC_WAVES, H, kinds), dim3(64 * CODEC_WAVES), 0, stream, A);
}

// Exclusive prefix sums of one head's tile sizes into off, and their total; called by all threads of a block, of which each SCAN_NT
// scan one list (tid: the thread's index among these; sh: one int per wave of the list).
constexpr int SCAN_NT = 512, SCAN_PER = 8;
__device__ __forceinline__ int scan_tile_bytes(const int* __restrict__ tb, int* __restrict__ off, int ntiles, int tid, int* sh) {
  const int wave = tid >> 6, lane = tid & 63;
  int carry = 0;
  for (int base = 0; base < ntiles; base += SCAN_NT * SCAN_PER) {
    const int t0 = base + tid * SCAN_PER;
    int n[SCAN_PER], mine = 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k) n[k] = tb[min(t0 + k, ntiles - 1)];
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k) { n[k] = t0 + k < ntiles ? n[k] : 0; mine += n[k]; }
    int incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(incl, o, 64); if (lane >= o) incl += v; }
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < SCAN_NT / 64; ++w) { const int v = sh[w]; all += v; before += w < wave ? v : 0; }
    int o = carry + before + incl - mine;
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k) { if (t0 + k < ntiles) off[t0 + k] = o; o += n[k]; }
    carry += all;
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
    if (host_bytes) host_bytes[h] = total;
  }
}

// Packs the per-tile escape slots into the heads' streams.  A block takes 64 consecutive tiles of a head, a wave 16 of them: the sizes and
// offsets of its tiles in one load each, then the first 64 bytes of all 16 slots in flight together (a tile has about 30 escape bytes;
// what is beyond 64 follows in a loop).  A wave that copied its tiles one after the other, each a chain of size -> bytes -> store, took
// 20.7 us for the 8 x 4096 tiles of a 64K-token page; this one takes 6.6 us and writes the row offsets as well (9.2 us of their own before).
// HEADS: the streams lie back to back and the block derives its head's start from the totals of the heads before it (a Page; it also
// writes head_start, the row offsets and the stream's padding); else head_start is given and a head whose window is too small is left out.
constexpr int PACK_TPB = 64;
struct PackKind { const uint8_t* slots; const int* tile_bytes; const int* tile_off; long off_stride; const int* head_start; uint8_t* ovf; };
struct PackArgs {
  PackKind j[2]; int ntiles;
  const int* head_bytes;                 // [kinds * H] totals (null without HEADS: every window is large enough)
  int window;                            // bytes that a head's stream must fit in (without HEADS)
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
  for (int k = 0; k < 16; ++k) v[k] = src[(long)min(t0 + k, A.ntiles - 1) * TILE_MAX_ESC + lane];
  long start = 0;
  if (HEADS) {
    __shared__ int part[4];
    int before = 0;
    for (int i = tid; i < h; i += 256) before += A.head_bytes[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    if (lane == 0) part[wave] = before;
    __syncthreads();
    start = part[0] + part[1] + part[2] + part[3];
    if (blockIdx.x == 0 && tid == 0) {
      A.head_start_out[h] = (int)start;
      if (h == H - 1) A.head_start_out[H] = (int)start + A.head_bytes[h];
    }
    if (blockIdx.x == 0 && h == H - 1 && tid < 8) J.ovf[start + A.head_bytes[h] + tid] = 0;      // readers fetch eight bytes at a time
  } else {
    if (A.head_bytes && A.head_bytes[(long)blockIdx.z * H + h] > A.window) return;
    start = J.head_start[h];
  }
  uint8_t* dst = J.ovf + start;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int n = __builtin_amdgcn_readlane(nb, k), o = __builtin_amdgcn_readlane(of, k);
    if (k >= n_own) break;
    if (lane < n) dst[o + lane] = (uint8_t)v[k];
    for (int i = 64 + lane; i < n; i += 64) dst[o + i] = src[(long)(t0 + k) * TILE_MAX_ESC + i];
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
// One wave per tile, four to a block: short-lived waves at full occupancy overlap the dependent loads of a tile (tag words -> escape
// bytes) with the arithmetic and the stores of others (four tiles in a row per wave were a third slower).
template <int KIND>
__global__ void __launch_bounds__(64) k_decode_tiles(const uint8_t* __restrict__ sm, const uint8_t* __restrict__ cd, const int* __restrict__ flags,
                                                     const int* __restrict__ tile_off, const uint8_t* __restrict__ ovf,
                                                     const int* __restrict__ head_start, const uint8_t* __restrict__ base3,
                                                     const uint8_t* __restrict__ base4, int n_kv, const int* __restrict__ bidx,
                                                     int S, int S_pad, u16* __restrict__ out, long out_head_stride, long out_row_stride) {
  const int tile = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int brow = bidx ? bidx[h] : h % n_kv;
  const long row0 = (long)h * S_pad + (long)tile * T;
  // rows beyond S carry tag 0 (the encoder writes every word of a tile) and are not written
  __shared__ __align__(16) u16 stage[T * STAGE_ROW];
  u16* dst = out + (long)h * out_head_stride + (long)tile * T * out_row_stride;
  const uint8_t* esc = ovf + head_start[h] + tile_off[(long)h * (S_pad / T) + tile];
  if ((out_row_stride & 7) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0)
    decode_tile_staged<KIND>(sm + row0 * D, cd + row0 * CB, flags + row0, esc, base3 + (long)brow * D, base4 + (long)brow * D, lane,
                             min(T, S - tile * T), stage, dst, out_row_stride);
  else      // rows that are not 16-byte aligned: element stores
    decode_tile_rows<KIND>(sm + row0 * D, cd + row0 * CB, flags + row0, esc, base3 + (long)brow * D, base4 + (long)brow * D, lane,
                           min(T, S - tile * T), dst, out_row_stride);
}

}  // namespace gaac

using namespace gaac;

extern "C" {

const char* gaac_last_error(void) { return last_error_buffer(); }

int gaac_exponent_hist(const void* x, long n_tokens, int n_kv, long long* hist, void* stream) {
  GAAC_REQUIRE(x && hist && n_kv > 0 && n_tokens >= 0, "gaac_exponent_hist: bad arguments");
  if (n_tokens == 0) return 0;
  int nchunk = (int)min((n_tokens + 1023) / 1024, 512L);
  int chunk = (int)((n_tokens + nchunk - 1) / nchunk);
  hipLaunchKernelGGL(k_exponent_hist, dim3(n_kv * D / HIST_CH, nchunk), dim3(256), 0, (hipStream_t)stream,
                     (const u16*)x, n_tokens, n_kv, chunk, (unsigned long long*)hist);
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
  launch_encode(A, H, 1, (hipStream_t)stream);
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
  A.head_bytes = head_bytes; A.flags = flags; A.S = S; A.S_pad = S_pad; A.head_start_out = head_start; A.ovf_off = ovf_off;
  hipLaunchKernelGGL(k_pack<true>, dim3((A.ntiles + PACK_TPB - 1) / PACK_TPB, H), dim3(256), 0, (hipStream_t)stream, A);
  return launch_status("gaac_page_pack");
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
  dim3 grid((S + T - 1) / T, H);
  if (kind == 0) hipLaunchKernelGGL(k_decode_tiles<KIND_K>, grid, dim3(64), 0, (hipStream_t)stream, sm, codes, flags, tile_off, ovf, head_start, base3, base4, n_kv, bidx, S, S_pad, (u16*)out, out_head_stride, out_row_stride);
  else hipLaunchKernelGGL(k_decode_tiles<KIND_V>, grid, dim3(64), 0, (hipStream_t)stream, sm, codes, flags, tile_off, ovf, head_start, base3, base4, n_kv, bidx, S, S_pad, (u16*)out, out_head_stride, out_row_stride);
  return launch_status("gaac_decode_tiles");
}

}  // extern "C"
