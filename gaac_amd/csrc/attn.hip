// Fused split-K decode attention over compressed K/V for gfx950 (wave64, MFMA), the raw-BF16 tail, and the split merge.
// Counterpart of gaac_attn / gaac_tail / gaac_combine / gaac_attn_launch in /root/reference/gaac/kernel.py:48-326
// (same inputs, same partial (m, l, acc) protocol, same slot map and padded-row behaviour), redesigned for CDNA4:
//
//   * one block = (batch row, kv head, split), 8 waves (one block per CU) for launches of up to 256 blocks, else 4 waves (two per CU);
//     the waves of a block take their tiles from a counter in LDS (the two waves sharing a SIMD would otherwise finish far apart);
//   * scores   S[16 tok x 16 heads]  = K[16 x 128] . Q^T      : 4 x v_mfma_f32_16x16x32_bf16   (A = decoded K units)
//   * output   O^T[128 x 16 heads]  += V^T[128 x 16] . P^T     : 8 x v_mfma_f32_16x16x16_bf16   (A = decoded V units)
//     The score tile lands in the register layout the second product wants for P^T, so P never crosses lanes.
//   * the GQA group (<= 16 query heads) rides in the N dimension; register use does not depend on it;
//   * three-stage prefetch per wave: tag words two tiles ahead, payload + escape bytes one tile ahead, consume;
//   * the raw BF16 tail of a cache head (<= 16 tokens) is attended by one wave of the block that owns the last split, as an extra
//     partial of that block's merge; the wave then joins the tile hand-out, so the other waves absorb the tiles it did not take;
//   * the last block of a (row, kv head) to publish its partial merges all of them (fused gaac_combine); k_attn_combine is the
//     two-launch alternative;
//   * k_attn_split<true, .> reads the paged slot pool through block and mode tables (paged_kernel.py:42-241).
//   Softmax runs in base 2 (scale * log2 e folded into the scores).
#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>
#include "gaac_tile.h"
#include "gaac_capi.h"
#include "../../include/gaac_hip.h"

// GAAC_WAVES12 (python -m gaac_amd.build --waves12 -> libgaac_hip_w12.so) is a measurement build, not the product: launches of up to
// 256 blocks over contiguous stores with host lengths run twelve-wave blocks, three waves per SIMD instead of two.  The register cap
// falls from 256 to 168 per lane; to get under it without spilling the tile loop, this build reads the query words from LDS for every
// score product instead of keeping them in 16 registers, and looks up the V side's escape and base words after the score products
// instead of together with the K side's.  Both cost time at two waves per SIMD, which is why the product does neither.
#ifdef GAAC_WAVES12
constexpr bool WAVES12 = true;
#else
constexpr bool WAVES12 = false;
#endif

namespace gaac {

constexpr int GMAX = 16;         // query heads per kv head the MFMA tile can carry
constexpr int MROW = D + 8;      // a head's accumulator row in the block merge: the heads of a store spread over the banks (in rows of 128 all heads of a store met in one: 16 query heads 14.4 -> 12.3 us)
constexpr int MAX_SLOTS = 1024;  // split partials a combine block can merge

struct StoreView {               // one kind (K or V) of a page or of a cache store
  const uint8_t* sm; const uint8_t* cd; const int* flags; const int* tile_off; const uint8_t* ovf; const int* head_start;
  const uint8_t* base3; const uint8_t* base4;
};
struct AttnArgs {
  StoreView k, v;
  const u16* q; float* pm; float* pl; float* pa;
  const int* slot; const int* sl;
  int S_pad; float scale_log2e; int nsplit; int nslot; int n_kv; int n_q; int G; int NB;
  const u16* kt; const u16* vt; const int* tl; int tcap;
  u32* epochs; u16* out;       // fused merge: [0] the epoch of the last merged launch, [1] failure bits, [2 + i] arrival mark of block i; pm / pl / pa then hold 64-bit records
  int S_all;                   // >= 0: every addressed cache head holds exactly S_all compressed tokens (sl is not read)
  // paged slot pool (k_attn_split<true>): sl = tokens per batch row, bt = block table [B][bt_stride], mt = mode table, pool = tile
  // slots of TS bytes, raw = side pool of BF16 tiles; physical tile = block*2*n_kv + 2*kvh + kind
  const uint8_t* pool; const u16* raw; const int* mt; const int* bt; int bt_stride; int TS;
  // paged: raw tiles queued by the preceding store (gaac_paged_store's freeq) that this launch pushes back onto the free stack (or null)
  const int* freeq; int n_free; int* stack; int* top;
  int B;                       // batch rows
  int plan;                    // > 0: the blocks share the rows out by length (plan_block), of which this many splits are resident at once; 0: nsplit blocks per row and kv head
#ifdef GAAC_PHASE_TIMING
  long long* dbg;
#endif
};
#ifdef GAAC_PHASE_TIMING
#define GAAC_STAMP(k) do { if (A.dbg && threadIdx.x == 0) A.dbg[(long)blockIdx.x * 8 + (k)] = wall_clock64(); } while (0)
#define GAAC_MSTAMP(k, v) do { if (A.dbg && threadIdx.x == 0) A.dbg[(2 * (long)gridDim.x + blockIdx.x) * 8 + (k)] = (v); } while (0)
#else
#define GAAC_STAMP(k) do {} while (0)
#define GAAC_MSTAMP(k, v) do {} while (0)
#endif
constexpr int MAX_CHUNK = 1024;  // tiles whose slot lookups a block keeps in LDS at a time (paged mode); longer splits go on in further rounds
constexpr int SLOT_CD = TILE_SM, SLOT_FL = TILE_SM + TILE_CD, SLOT_OV = SLOT_FL + 4 * T;      // byte offsets inside a tile slot

// n / d for the block's own coordinates: the compiler's 32-bit division is a chain of quarter-rate multiplications, and a block needs five
// quotients before it can load anything.  Below 2^21 the rounded product is exact: (n + 0.5) / d is at least 0.5 / d away from an
// integer, the product is off by less than 2^-22 n / d.
constexpr int SMALL_DIV = 1 << 21;
__device__ __forceinline__ int div_below_2_21(int n, int d) { return (int)(((float)n + 0.5f) * __builtin_amdgcn_rcpf((float)d)); }
__device__ __forceinline__ int small_div(int n, int d) {
  if (__builtin_expect(n >= SMALL_DIV, 0)) return n / d;
  return div_below_2_21(n, d);
}
__device__ __forceinline__ float bf16_bits_to_float(u32 h) { return __uint_as_float(h << 16); }
__device__ __forceinline__ u32 pack_bf16x2(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  bf16x2 v; v[0] = (__bf16)lo; v[1] = (__bf16)hi;
  return __builtin_bit_cast(u32, v);
}

// ---------------------------------------------------------------------------------------------------- fused merge
// Merge of the split partials (gaac_combine, /root/reference/gaac/kernel.py:281-294) inside the split kernel, by ONE block of each
// (batch row, kv head), without atomics and without any block waiting for a store acknowledgement on its way out:
//
//   * One word, epochs[0], holds the epoch of the last merged launch.  Every block reads it while its first tiles are in flight; this
//     launch's EPOCH is that value + 1 (skipping 0 when the 32-bit counter wraps), the same for all blocks: the word is advanced by
//     the last block of the grid, as its very last action, and only after it has SEEN the arrival mark of every block of the grid
//     (epochs[2 + block], stored by the block once its first wave is through its tiles: a block that has marked has read the word
//     long ago; blocks of a grid larger than the GPU holds start whenever a CU of their XCD frees up, in no order the other XCDs
//     know of).
//     A record slot read by a launch was last written by an earlier launch, whatever its shape, under another epoch (the same
//     value returns only after 2^32 - 1 launches on the same records), or never, and then holds the unused epoch 0.
//   * A partial value travels as one 64-bit record (fp32 bits | epoch << 32) written with a single 64-bit store: a reader sees either
//     the whole record of this launch or an older one, never a torn one (naturally aligned 64-bit accesses are single-copy atomic),
//     so no fence, flag or acknowledgement orders data against a separate signal.  Records are written with agent-scope stores
//     (write-through) and read with agent-scope loads (they bypass the reader's L2): the blocks of a head sit on different XCDs.
//   * The MERGERS are the head's last (up to sixteen) blocks in index order; each takes a share of the head's output (half a query head
//     per wave), because one CU pulls records at only ~80 GB/s.  Once a merger has stored its own partial it loads the records of its
//     share from all blocks of the head and re-reads those whose epoch is not yet the launch's.  Everything a merger waits for is
//     running, done, or one of the at most fifteen later mergers of the same head, which wait for nobody but each other's stores,
//     and those precede every wait.  The wait is bounded all the same (MERGE_SPIN_LIMIT re-reads): a merger that gives up writes its
//     rows as NaN and sets bit 0 of epochs[1].  The grid's last block may have little or nothing to do of its own (a short row; no unit left
//     for it in a planned launch) and then waits for the whole launch: its bound (EPOCH_SPIN_LIMIT) is some seconds, far above any
//     launch.  It sets bit 1 if it gives up (and leaves the epoch word alone).  The owner of the workspace polls epochs[1] and re-arms
//     after a failure.
//   * Launches that share the records and the epoch words must be ordered on one stream.  To re-arm after a failed launch, zero all.
typedef __attribute__((ext_vector_type(4))) float f32x4v;
__device__ __forceinline__ void store_partial(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void ll_store(u64* p, float v, u32 epoch) {
  __hip_atomic_store(p, (u64)__float_as_uint(v) | ((u64)epoch << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 ll_load(const u64* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ bool ll_stale(u64 r, u32 epoch) { return (u32)(r >> 32) != epoch; }
__device__ __forceinline__ float ll_value(u64 r) { return __uint_as_float((u32)r); }
constexpr int MERGE_SPIN_LIMIT = 1 << 16;      // re-reads of a chunk before the merger gives up (each with a short sleep: ~0.1 s)
constexpr int EPOCH_SPIN_LIMIT = 1 << 23;      // polls of the arrival marks before the grid's last block gives up (about a microsecond each)
// (no branch around the load: a load under a branch is waited for where the branch ends, together with everything issued before it)
__device__ __forceinline__ u32 load_epoch(const AttnArgs& A) {
  const u32* p = A.epochs ? A.epochs : reinterpret_cast<const u32*>(A.q);
  const u32 e = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return e + 1u + (e == 0xFFFFFFFFu ? 1u : 0u);      // epoch 0 is never used: zeroed records stay stale when the counter wraps
}
// A block barrier that orders LDS traffic only.  (__syncthreads() also waits for the block's global stores to be acknowledged,
// which for write-through stores is a trip to memory.)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// LDS of a merging block: per wave the (m, then weight) and l of every slot.
template <int NW> struct MergeScratch { float f[NW][MAX_SLOTS], l[NW][MAX_SLOTS]; };

// One merger's work for half a query head (64 output channels), shared by NW waves (of the block, or half the block's: see merge_heads), of which
// this is the wave-th; fs, ls: its own part of the scratch.  A wave owns 64 / NW channels
// and sums them over ALL slots, so the waves exchange nothing and no block barrier lies between the records' arrival and the
// output: lane (g, c) = (lane / CPW, lane % CPW) reads the accumulator records of channel c of the wave for the slots g, g + SG, ...
// (SG = 64 / CPW slot groups); the groups' sums meet through DPP.  Every wave reads the m / l records of all slots (lane = slot)
// and derives the slots' weights itself.  rec: the query head's first record, nslot: its splits.  Called by all threads of the block.
__device__ __forceinline__ void merge_failed(const AttnArgs& A, u32 bit) {
  __hip_atomic_fetch_or(A.epochs + 1, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int NW>
__device__ __forceinline__ void merge_half_head(const AttnArgs& A, long rec, int nslot, long row, int half, u32 epoch, float* fs, float* ls, int wave, int lane) {
  constexpr int CPW = 64 / NW, SG = 64 / CPW;      // channels per wave (8 | 16), slot groups (8 | 4)
  constexpr int CH = 8;                             // accumulator records in flight per lane: one round for up to CH * SG splits
  const int g = lane / CPW, d0 = 64 * half + CPW * wave, d = d0 + lane % CPW;
  const u64* rm = reinterpret_cast<const u64*>(A.pm) + rec;
  const u64* rl = reinterpret_cast<const u64*>(A.pl) + rec;
  // (a uniform base and a 32-bit offset per lane, at most (MAX_SLOTS - 1) * D + 15 records: the addresses of the first round's loads are
  // on the way of every launch.  With 64-bit addresses per lane a launch took 0.05-0.2 us more: 2 rows x 4096 tokens 11.64 against 11.45)
  const u64* ra0 = reinterpret_cast<const u64*>(A.pa) + rec * D + d0;
  const u64* ra = ra0 + lane % CPW;
  bool ok = true;
  // all loads of the first round are issued before the first use, none under a branch (a slot past the end reads the last slot
  // instead and is ignored): the lane's first CH accumulator records ...
  u64 v[CH];
#pragma unroll
  for (int k = 0; k < CH; ++k) v[k] = ll_load(ra0 + ((u32)min(g + SG * k, nslot - 1) * D + (u32)(lane % CPW)));
  // ... then m / l of slots 0..63 (one slot per lane); everything is re-read together until it carries this launch's epoch
  u64 mr = ll_load(rm + (u32)min(lane, nslot - 1)), lr = ll_load(rl + (u32)min(lane, nslot - 1));
  GAAC_MSTAMP(0, wall_clock64());
  for (int spin = 0;; ++spin) {
    bool stale = lane < nslot && (ll_stale(mr, epoch) || ll_stale(lr, epoch));
#pragma unroll
    for (int k = 0; k < CH; ++k) stale |= g + SG * k < nslot && ll_stale(v[k], epoch);
    if (__builtin_amdgcn_ballot_w64(stale) == 0) break;
    if (spin >= MERGE_SPIN_LIMIT) { ok = false; break; }
    __builtin_amdgcn_s_sleep(1);
    if (lane < nslot && ll_stale(mr, epoch)) mr = ll_load(rm + lane);
    if (lane < nslot && ll_stale(lr, epoch)) lr = ll_load(rl + lane);
#pragma unroll
    for (int k = 0; k < CH; ++k) { const int s = g + SG * k; if (s < nslot && ll_stale(v[k], epoch)) v[k] = ll_load(ra + (long)s * D); }
  }
  GAAC_MSTAMP(1, wall_clock64());
  const float m_own = lane < nslot ? ll_value(mr) : -INFINITY, l_own = lane < nslot ? ll_value(lr) : 0.f;      // slot = lane
  float m = m_own;
  for (int s0 = 64; ok && s0 < nslot; s0 += 64) {      // more than 64 splits: the other m / l records, kept in LDS
    const int s = s0 + lane;
    mr = s < nslot ? ll_load(rm + s) : 0ull; lr = s < nslot ? ll_load(rl + s) : 0ull;
    for (int spin = 0; __builtin_amdgcn_ballot_w64(s < nslot && (ll_stale(mr, epoch) || ll_stale(lr, epoch))) != 0; ++spin) {
      if (spin >= MERGE_SPIN_LIMIT) { ok = false; break; }
      __builtin_amdgcn_s_sleep(1);
      if (s < nslot && ll_stale(mr, epoch)) mr = ll_load(rm + s);
      if (s < nslot && ll_stale(lr, epoch)) lr = ll_load(rl + s);
    }
    if (s < nslot) { fs[s] = ll_value(mr); ls[s] = ll_value(lr); m = fmaxf(m, ll_value(mr)); }
  }
  const float mx = wave_max(m);
  // the slots' weights go to LDS for the lanes that need them (the wave's own region: no block barrier)
  const float f_own = m_own != -INFINITY ? __builtin_amdgcn_exp2f(m_own - mx) : 0.f;
  float l = l_own * f_own;
  fs[lane] = f_own;
  for (int s = lane + 64; s < nslot; s += 64) {      // each lane revisits the slots it wrote
    const float pmv = fs[s], f = pmv != -INFINITY ? __builtin_amdgcn_exp2f(pmv - mx) : 0.f;
    fs[s] = f; l += ls[s] * f;
  }
  wave_lds_sync();
  // The weights of the lane's first round in one batch of reads, none under a branch (slots past the end weigh 0).  Read one after the other
  // where they are used, eight trips through LDS, they made the sums 0.65 to 0.8 us of the launch; now 0.4: 64K tokens x 4 kv heads of 6 query heads
  // 22.8 -> 22.3 us, 1000 x 8 8.2 -> 8.0, 4000 x 1 of 16 10.7 -> 10.1.
  float f[CH];
#pragma unroll
  for (int k = 0; k < CH; ++k) f[k] = fs[g + SG * k];
  l = wave_sum(l);
  float acc = 0.f;
#pragma unroll
  for (int k = 0; k < CH; ++k) acc += f[k] != 0.f ? ll_value(v[k]) * f[k] : 0.f;      // an empty partial's accumulator may hold anything
  for (int s0 = g + SG * CH; s0 < nslot; s0 += SG * CH) {      // more than CH * SG splits: the lane's further records
#pragma unroll
    for (int k = 0; k < CH; ++k) { const int s = s0 + SG * k; v[k] = s < nslot ? ll_load(ra + (long)s * D) : 0ull; }
    for (int spin = 0; ok; ++spin) {
      bool stale = false;
#pragma unroll
      for (int k = 0; k < CH; ++k) stale |= s0 + SG * k < nslot && ll_stale(v[k], epoch);
      if (__builtin_amdgcn_ballot_w64(stale) == 0) break;
      if (spin >= MERGE_SPIN_LIMIT) { ok = false; break; }
      __builtin_amdgcn_s_sleep(1);
#pragma unroll
      for (int k = 0; k < CH; ++k) { const int s = s0 + SG * k; if (s < nslot && ll_stale(v[k], epoch)) v[k] = ll_load(ra + (long)s * D); }
    }
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int s = s0 + SG * k;
      if (s < nslot) { const float fk = fs[s]; acc += fk != 0.f ? ll_value(v[k]) * fk : 0.f; }
    }
  }
  // the slot groups' sums of a channel sit CPW lanes apart: across the four 16-lane rows, and for CPW = 8 also 8 lanes apart in a row
  acc = quad_rows_sum(acc);
  if (CPW == 8) acc += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, acc), 0x128 /* row_ror:8 */, 0xF, 0xF, false));
  GAAC_MSTAMP(2, wall_clock64());
  ok = __builtin_amdgcn_ballot_w64(!ok) == 0;
  if (!ok && lane == 0) merge_failed(A, 1u);
  if (lane < CPW) {
    const float o = ok ? (l > 0.f ? acc / l : 0.f) : __builtin_nanf("");
    A.out[row * D + d] = __builtin_bit_cast(u16, (__bf16)o);
  }
  GAAC_MSTAMP(4, wall_clock64());
  wave_lds_sync();      // the wave's LDS region is free for its next item
}
// The same for a head of at most WAVE_MERGE_SLOTS splits, and of fewer splits than half heads, by ONE wave: lane = channel, all records of
// the half head in flight together.  With few splits there are few mergers, and a block that works on one half head at a time pays a trip
// to memory for each (2 splits and 4 query heads: four in a row): here each wave of the merging blocks takes a half head of its own.
// Launches over 1000 tokens x 8 kv heads, block-wise -> wave-wise: 18.1 -> 13.2 us with two splits, 15.1 -> 11.3 with three, 12.8 -> 10.6
// with four, 11.1 -> 9.0 with six; 4000 tokens, 1 kv head with 16 query heads: 20.4 -> 15.9 with nine, 18.2 -> 14.8 with twelve, 15.8 -> 13.8
// with sixteen, which is as many as a lane keeps records for; 2 kv heads with 8: 15.6 -> 13.5 with nine, 13.0 -> 11.6 with fifteen.
// With as many splits as half heads each merging block has one half head, a single trip as well, and spreads its records over more waves.
constexpr int WAVE_MERGE_SLOTS = 16;
template <int SLOTS>      // how many it reads (those past the last split again: no load under a branch)
__device__ __forceinline__ void merge_half_head_wave(const AttnArgs& A, long rec, int nslot, long row, int half, u32 epoch, int lane) {
  const int d = 64 * half + lane;
  const u64* rm = reinterpret_cast<const u64*>(A.pm) + rec + min(lane, nslot - 1);
  const u64* rl = reinterpret_cast<const u64*>(A.pl) + rec + min(lane, nslot - 1);
  const u64* ra = reinterpret_cast<const u64*>(A.pa) + rec * D + d;
  u64 v[SLOTS];
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) v[k] = ll_load(ra + (long)min(k, nslot - 1) * D);      // (past the end: the last record again, ignored)
  u64 mr = ll_load(rm), lr = ll_load(rl);
  bool ok = true;
  for (int spin = 0;; ++spin) {
    bool stale = ll_stale(mr, epoch) || ll_stale(lr, epoch);
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) stale |= ll_stale(v[k], epoch);
    if (__builtin_amdgcn_ballot_w64(stale) == 0) break;
    if (spin >= MERGE_SPIN_LIMIT) { ok = false; break; }
    __builtin_amdgcn_s_sleep(1);
    if (ll_stale(mr, epoch)) mr = ll_load(rm);
    if (ll_stale(lr, epoch)) lr = ll_load(rl);
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) if (ll_stale(v[k], epoch)) v[k] = ll_load(ra + (long)min(k, nslot - 1) * D);
  }
  const float m = lane < nslot ? ll_value(mr) : -INFINITY, mx = wave_max(m);
  const float f = m != -INFINITY ? __builtin_amdgcn_exp2f(m - mx) : 0.f;      // 0 also for the lanes without a slot
  const float l = wave_sum(ll_value(lr) * f);
  float acc = 0.f;
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) {
    const float fk = __uint_as_float((u32)__builtin_amdgcn_readlane((int)__float_as_uint(f), k));
    acc += fk != 0.f ? ll_value(v[k]) * fk : 0.f;      // an empty partial's accumulator may hold anything
  }
  if (!ok && lane == 0) merge_failed(A, 1u);
  A.out[row * D + d] = __builtin_bit_cast(u16, (__bf16)(ok ? (l > 0.f ? acc / l : 0.f) : __builtin_nanf("")));
}
// The merge of a head is shared by its last `mergers` blocks in index order (merge_ranks): the block of rank j takes the half heads
// j, j + mergers, ..., so that no single CU has to pull all the records; a head with fewer splits than half heads, and few of them,
// is merged wave by wave.  Called by all threads of a merging block after its own partial has been stored and every thread is done
// with the LDS that X aliases.
__device__ __forceinline__ int merge_ranks(int G, int nslot) { return min(min(16, 2 * G), nslot); }
// Arrival marks: epochs[2 + i] = the epoch block i of the grid works under, stored by the block's first wave when it leaves its tile
// loop (long after it read the epoch word, well before the block publishes its partial).  The grid's last block reads all marks
// before it advances the epoch word.
constexpr int EPOCH_WORDS = 2;      // words of the epoch buffer ahead of the arrival marks
__device__ __forceinline__ void mark_arrival(const AttnArgs& A, u32 epoch) {
  __hip_atomic_store(A.epochs + EPOCH_WORDS + blockIdx.x, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The grid's last block advances the epoch word for the next launch, once every block of this launch has marked its arrival (and so has
// read the word).  Where the block has merge work, the marks' first read (the first 2048 blocks) is issued ahead of it and looked at after it: by
// then the other blocks of an evenly shared launch have long left their loops, so the check normally costs no trip to memory of its own.
template <int NW> struct MarkRegs { u32 m[2048 / (64 * NW)]; };
template <int NW>
__device__ __forceinline__ void load_marks(const AttnArgs& A, int tid, MarkRegs<NW>& R) {
#pragma unroll
  for (int k = 0; k < 2048 / (64 * NW); ++k)
    R.m[k] = __hip_atomic_load(A.epochs + EPOCH_WORDS + min(tid + 64 * NW * k, (int)gridDim.x - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int NW>      // called by NW waves of the block; verdict: one word of LDS per wave
__device__ __forceinline__ void advance_epoch(const AttnArgs& A, u32 epoch, int tid, MarkRegs<NW>& R, float* verdict, int verdict_stride) {
  constexpr int XK = 2048 / (64 * NW);
  const u32* marks = A.epochs + EPOCH_WORDS;
  const int nblocks = (int)gridDim.x, wave = tid >> 6, lane = tid & 63;
  bool grid_ok = true;
  for (int spin = 0;; ++spin) {
    bool stale = false;
#pragma unroll
    for (int k = 0; k < XK; ++k) stale |= R.m[k] != epoch;
    if (__builtin_amdgcn_ballot_w64(stale) == 0) break;
    if (spin >= EPOCH_SPIN_LIMIT) { grid_ok = false; break; }
    __builtin_amdgcn_s_sleep(1);
#pragma unroll
    for (int k = 0; k < XK; ++k)
      if (R.m[k] != epoch) R.m[k] = __hip_atomic_load(marks + min(tid + 64 * NW * k, nblocks - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  for (int i0 = 2048; grid_ok && i0 < nblocks; i0 += 64 * NW) {      // grids beyond 2048 blocks: the remaining marks, a round at a time
    const int i = min(i0 + tid, nblocks - 1);
    for (int spin = 0; __builtin_amdgcn_ballot_w64(__hip_atomic_load(marks + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != epoch) != 0; ++spin) {
      if (spin >= EPOCH_SPIN_LIMIT) { grid_ok = false; break; }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  // The waves' verdicts meet in LDS behind a barrier that orders LDS traffic only: a full block barrier would first wait for the
  // acknowledgement of the output rows just stored, and the epoch store would then be a second trip to memory at the launch's very end.
  grid_ok = __builtin_amdgcn_ballot_w64(!grid_ok) == 0;
  if (lane == 0) verdict[wave * verdict_stride] = grid_ok ? 1.f : 0.f;
  lds_barrier();
  if (tid == 0) {
    bool all = true;
#pragma unroll
    for (int w = 0; w < NW; ++w) all &= verdict[w * verdict_stride] != 0.f;
    if (all) __hip_atomic_store(A.epochs, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else merge_failed(A, 2u);
  }
}
// rec0: the first record of query head 0 of the group, nslot: the splits of the head, rank < 0 or nslot 1: nothing to merge here.
template <int NWB>      // NWB: waves of the block; twelve-wave blocks (measurement build) merge with their first eight waves
__device__ __forceinline__ void merge_heads(const AttnArgs& A, long qh0, int G, u32 epoch, long rec0, int nslot, int rank, int mergers, int tid, MergeScratch<(NWB > 8 ? 8 : NWB)>& X) {
  constexpr int NW = NWB > 8 ? 8 : NWB;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  if (NWB > NW && wave >= NW) { if (blockIdx.x == gridDim.x - 1) lds_barrier(); return; }      // (the last block meets once more below)
  const bool last = blockIdx.x == gridDim.x - 1;
  MarkRegs<NW> xm;
  if (last) load_marks<NW>(A, tid, xm);
  // The first item stands outside the loop: at a loop header the compiler waits for every memory operation in flight, which here
  // would be the acknowledgement of the block's own record stores (a round trip to memory) before the first record load is issued.
  if (rank >= 0 && nslot > 1) {
    if (nslot <= WAVE_MERGE_SLOTS && nslot < 2 * G) {
      // (a wave has one item, or two at sixteen query heads and two splits)
      for (int item = rank + mergers * wave; item < 2 * G; item += mergers * NW) {
        if (nslot <= 8) merge_half_head_wave<8>(A, rec0 + (long)(item >> 1) * nslot, nslot, qh0 + (item >> 1), item & 1, epoch, lane);
        else merge_half_head_wave<WAVE_MERGE_SLOTS>(A, rec0 + (long)(item >> 1) * nslot, nslot, qh0 + (item >> 1), item & 1, epoch, lane);
      }
    } else if (NW == 8 && 2 * G > mergers) {
      // more half heads than mergers (nine query heads and up): the block's halves take one each.  One after the other they were two trips to
      // memory: 1 kv head of 16 query heads, 2000 tokens in 32 splits 11.7 -> 9.9 us, 6000 in 64 12.2 -> 11.6, slot cache 790 in 25 12.5 -> 10.8
      const int item = rank + mergers * (wave >> 2);
      if (item < 2 * G) merge_half_head<4>(A, rec0 + (long)(item >> 1) * nslot, nslot, qh0 + (item >> 1), item & 1, epoch, X.f[wave], X.l[wave], wave & 3, lane);
    } else {
      int item = rank;
      if (item < 2 * G) { merge_half_head<NW>(A, rec0 + (long)(item >> 1) * nslot, nslot, qh0 + (item >> 1), item & 1, epoch, X.f[wave], X.l[wave], wave, lane); item += mergers; }
      for (; item < 2 * G; item += mergers) merge_half_head<NW>(A, rec0 + (long)(item >> 1) * nslot, nslot, qh0 + (item >> 1), item & 1, epoch, X.f[wave], X.l[wave], wave, lane);
    }
  }
  if (last) advance_epoch<NW>(A, epoch, tid, xm, &X.l[0][0], MAX_SLOTS);
}

// ---------------------------------------------------------------------------------------------------- uncompressed rows
// Attention of the block's query heads over up to 16 rows kept as plain BF16: the raw tail of a cache head (gaac_tail of
// /root/reference/gaac/kernel.py:220-279) or a raw tile of the paged pool.  ONE wave does it, ahead of its tiles, and the block's other
// waves take the tiles that it does not get to.  All rows and queries are loaded in one batch, so it costs one trip to memory and some
// 60 matrix products however many query heads there are; weights and sums stay in fp32:
//   * scores: 4 x v_mfma_f32_16x16x32_bf16 over the rows as they lie (products of BF16 are exact in fp32), lane (head a, quad q) gets tokens 4q + r;
//   * output: 32 x v_mfma_f32_16x16x4_f32; its B operand is the weight p[r] where the score product left it, A the V row 4q + r in fp32.
// Before, in vector arithmetic with a trip to memory per query head for its queries: 3 us beyond the tiles of the block with 4 query heads, 10
// with 16, at the end of which the launch waited; a raw tile of the paged pool was taken by the whole block behind its tiles, through six
// barriers, one of which every block of the launch paid for.  Launches in a graph, us: slot cache, 4 rows of 790 tokens x 8 kv heads x 4 query
// heads 11.1 -> 9.8, 1 row x 1 kv head x 16 21.0 -> 13.6; paged, 8 sequences of 200..3000 x 8 kv heads 24.0 -> 21.7, 16 of 32000 276 -> 249,
// 16 of 4096..65536 297 -> 284, 1 of 900 x 1 kv head x 16 29.0 -> 19.0.
struct RawState { f32x4 acc[8]; float m, l; };      // acc[i][r] = O[head a][channel 8 (4q + r) + i]; m in the base-2 domain
// krows / vrows: rows of 128 BF16 back to back, of which the first nvalid (1..16) count; qr[j]: channels 32j + 8q .. + 8 of query head a
__device__ __forceinline__ void raw_rows_attend(const u16* krows, const u16* vrows, int nvalid, const u32x4 (&qr)[4], float scale_log2e, int a, int q, RawState& st) {
  u32x4 k[4], v[4];      // no load under a branch: rows past the end read the last valid row
#pragma unroll
  for (int j = 0; j < 4; ++j) k[j] = *reinterpret_cast<const u32x4*>(krows + min(a, nvalid - 1) * D + 32 * j + 8 * q);
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = *reinterpret_cast<const u32x4*>(vrows + min(4 * q + r, nvalid - 1) * D + 8 * a);
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k[j]), __builtin_bit_cast(bf16x8, qr[j]), s, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) s[r] = 4 * q + r < nvalid ? s[r] * scale_log2e : -INFINITY;
  const float m = fmaxf(st.m, quad_rows_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])))), mu = m == -INFINITY ? 0.f : m;
  const float alpha = st.m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(st.m - mu);
  float p[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(s[r] - mu);      // rows past the end: exp2(-inf) = 0
  st.m = m; st.l = st.l * alpha + quad_rows_sum((p[0] + p[1]) + (p[2] + p[3]));
#pragma unroll
  for (int i = 0; i < 8; ++i) st.acc[i] *= alpha;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const bool there = 4 * q + r < nvalid;      // rows past the end weigh 0: keep an Inf of the clamped row out of 0 * Inf
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32 w = there ? v[r][i] : 0u;
      st.acc[2 * i] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf16_bits_to_float(w & 0xFFFFu), p[r], st.acc[2 * i], 0, 0, 0);
      st.acc[2 * i + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w & 0xFFFF0000u), p[r], st.acc[2 * i + 1], 0, 0, 0);
    }
  }
}
__device__ __forceinline__ void raw_queries(const u16* qrows, int G, int a, int q, u32x4 (&qr)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) qr[j] = *reinterpret_cast<const u32x4*>(qrows + min(a, G - 1) * D + 32 * j + 8 * q);      // (heads past the last: any valid row)
}
// the result as one more partial of the block's merge: m, l [GMAX], acc [GMAX][D]
__device__ __forceinline__ void raw_rows_store(const RawState& st, int a, int q, float* __restrict__ m, float* __restrict__ l, float (*__restrict__ acc)[MROW]) {
  if (q == 0) { m[a] = st.m; l[a] = st.l; }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float* o = &acc[a][8 * (4 * q + r)];
    *reinterpret_cast<f32x4*>(o) = f32x4{st.acc[0][r], st.acc[1][r], st.acc[2][r], st.acc[3][r]};
    *reinterpret_cast<f32x4*>(o + 4) = f32x4{st.acc[4][r], st.acc[5][r], st.acc[6][r], st.acc[7][r]};
  }
}
// ... and back, for a block that meets further raw rows
__device__ __forceinline__ void raw_rows_load(RawState& st, int a, int q, const float* __restrict__ m, const float* __restrict__ l, const float (*__restrict__ acc)[MROW]) {
  st.m = m[a]; st.l = l[a];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) st.acc[i][r] = st.m == -INFINITY ? 0.f : acc[a][8 * (4 * q + r) + i];      // (none yet: may hold anything)
}

// ---------------------------------------------------------------------------------------------------- block tables (LDS)
// xlut[e]: the four exponent-field words carrying the 4th code bits of escape byte e (bit p -> element p, bit 4+p -> element p+4).
// sel[t]:  v_perm selector that spreads a lane's 8 prefetched escape bytes to one byte per unit, indexed by the lane's four
//          tags t (2 bits each): byte u = offset of unit u's escape byte when the unit is a 4-bit group (and the offset
//          is < 8), else 0x0C (-> 0).
// bw*:     exponent-base words [tier][group][p] of this block's kv head;  qw: the query words [head][group][p].
struct AttnLds {
  u32x4 xlut[256];
  u32 sel[256];
  u32x4 bwk[2][NG], bwv[2][NG];
  u32x4 qw[GMAX][NG];
};
// Block merge: one partial per wave plus one or two (index NW) for the uncompressed rows.  Before the waves publish, a wave w that takes these keeps the
// decoded side of a half raw tile in acc[w]; afterwards the mergers' scratch lies in acc.
// RAWS: waves that take uncompressed rows, a partial each.
template <int NW, int RAWS> struct MergeLds { float m[NW + RAWS][GMAX], l[NW + RAWS][GMAX]; __align__(16) float acc[NW + RAWS][GMAX][MROW]; };
static_assert(T * D * sizeof(u16) <= GMAX * D * sizeof(float) && sizeof(MergeScratch<4>) <= 5 * GMAX * D * sizeof(float) &&
              sizeof(MergeScratch<8>) <= 9 * GMAX * D * sizeof(float), "scratch views must fit the merge buffer");
struct TableRegs { u32 b0, b1; u32 qlo[4], qhi[4]; };      // one thread's raw inputs of the per-block tables
// Global loads only, in two parts so that each can be issued as soon as its address is known (the query rows need the batch row, the
// base rows the cache head) and waited for only when the tables are written.
__device__ __forceinline__ void tables_load_q(TableRegs& Tr, int tid, const u16* __restrict__ qrows, int G) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {      // query words: head = idx >> 6, group = (idx >> 2) & 15, p = idx & 3 (heads >= G: any valid row)
    const int idx = tid + 256 * k, h = min(idx >> 6, G - 1), g = (idx >> 2) & 15, p = idx & 3;
    const u16* qp = qrows + h * D;
    Tr.qlo[k] = qp[chan_k(8 * g + p)]; Tr.qhi[k] = qp[chan_k(8 * g + p + 4)];
  }
}
__device__ __forceinline__ void tables_load_bases(TableRegs& Tr, int tid, const uint8_t* k3, const uint8_t* k4, const uint8_t* v3,
                                                  const uint8_t* v4, int brow) {
  // one base word per thread: kind = tid >> 7, tier = (tid >> 6) & 1, group = (tid >> 2) & 15, p = tid & 3
  const int kind = tid >> 7, tier = (tid >> 6) & 1, g = (tid >> 2) & 15, p = tid & 3;
  const uint8_t* row = (kind ? (tier ? v4 : v3) : (tier ? k4 : k3)) + (long)brow * D;
  const int c0 = kind ? chan_v(8 * g + p) : chan_k(8 * g + p), c1 = kind ? chan_v(8 * g + p + 4) : chan_k(8 * g + p + 4);
  Tr.b0 = row[c0]; Tr.b1 = row[c1];
}
__device__ __forceinline__ void tables_store(AttnLds& L, TableRegs Tr, int tid, int G) {
  // the loaded values are first needed HERE: keeps the compiler from packing them (and waiting for them) where they were loaded
  asm volatile("" : "+v"(Tr.b0), "+v"(Tr.b1), "+v"(Tr.qlo[0]), "+v"(Tr.qlo[1]), "+v"(Tr.qlo[2]), "+v"(Tr.qlo[3]), "+v"(Tr.qhi[0]),
               "+v"(Tr.qhi[1]), "+v"(Tr.qhi[2]), "+v"(Tr.qhi[3]));
  {
    const u32 e = (u32)tid;
    u32x4 w;
#pragma unroll
    for (int p = 0; p < 4; ++p) w[p] = (((e >> p) & 1u) << 10) | (((e >> (4 + p)) & 1u) << 26);
    L.xlut[tid] = w;
    u32 selw = 0u, off = 0u;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const u32 t = (e >> (2 * u)) & 3u;
      selw |= ((t == 1u && off < 8u) ? off : 0x0Cu) << (8 * u);
      off += (u32)tag_size(t);
    }
    L.sel[tid] = selw;
  }
  {
    const int kind = tid >> 7, tier = (tid >> 6) & 1, g = (tid >> 2) & 15, p = tid & 3;
    u32* dst = kind ? reinterpret_cast<u32*>(&L.bwv[tier][g]) : reinterpret_cast<u32*>(&L.bwk[tier][g]);
    dst[p] = (Tr.b0 << 7) | (Tr.b1 << 23);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int idx = tid + 256 * k, h = idx >> 6, g = (idx >> 2) & 15, p = idx & 3;
    reinterpret_cast<u32*>(&L.qw[h][g])[p] = h < G ? Tr.qlo[k] | (Tr.qhi[k] << 16) : 0u;
  }
}

// ---------------------------------------------------------------------------------------------------- tile loaders
struct KindRegs {                // one lane's view of one tile (K or V)
  Payload pay;
  u32 f;                         // the lane's four tags (bits 8q .. 8q+7 of the tag word of its line)
  u32 pos0;                      // offset of the lane's first unit's escape bytes: in the head's stream | in the tile (paged)
  u32x2 e;                       // the 8 escape bytes from pos0 on
};
struct TileRegs { KindRegs k, v; };
struct TagRegs { u32 kfl, vfl; u32 kto, vto; int raw; };      // kto/vto: tile offset in the head's escape stream | slot index (paged)

struct Bases {                   // uniform (scalar) views of one cache head; paged mode uses kov = vov = pool and TS only
  const uint8_t* ksm; const uint8_t* kcd; const int* kfl; const int* kto; const uint8_t* kov;
  const uint8_t* vsm; const uint8_t* vcd; const int* vfl; const int* vto; const uint8_t* vov;
  int TS;
};
struct TileTable { const int2* tt; int tlo; };      // paged mode: mode-table entries (K, V) of the block's tiles, in LDS

// start of a tile's escape bytes
template <bool PAGED>
__device__ __forceinline__ const uint8_t* esc_of_tile(const uint8_t* ov, u32 to, int TS) {
  return PAGED ? ov + (size_t)to * (size_t)TS + SLOT_OV : ov + to;
}

template <bool PAGED>
__device__ __forceinline__ void load_tags(const Bases& B, const TileTable& TT, int tile, int a, TagRegs& Tg) {
  if (PAGED) {
    const int2 e = TT.tt[tile - TT.tlo];
    const int ek = __builtin_amdgcn_readfirstlane(e.x), ev = __builtin_amdgcn_readfirstlane(e.y);
    Tg.raw = (ek | ev) < 0;                       // a tile with a raw side is skipped here, see attend_raw_tiles
    Tg.kto = (u32)max(ek, 0); Tg.vto = (u32)max(ev, 0);
    Tg.kfl = reinterpret_cast<const u32*>(B.kov + (size_t)Tg.kto * (size_t)B.TS + SLOT_FL)[a];
    Tg.vfl = reinterpret_cast<const u32*>(B.vov + (size_t)Tg.vto * (size_t)B.TS + SLOT_FL)[a];
  } else {
    const u32 w = (u32)(tile * T + a);
    Tg.kfl = (u32)__builtin_nontemporal_load(B.kfl + w); Tg.vfl = (u32)__builtin_nontemporal_load(B.vfl + w);
    Tg.kto = (u32)B.kto[(u32)tile]; Tg.vto = (u32)B.vto[(u32)tile];
    Tg.raw = 0;
  }
}

// the tile's sign/mantissa and code bytes (paged mode: the slot index comes with the tags)
template <bool PAGED>
__device__ __forceinline__ void load_tile_payload(const Bases& B, int tile, int lane, const TagRegs& Tg, TileRegs& R) {
  if (PAGED) {
    const uint8_t* ks = B.kov + (size_t)__builtin_amdgcn_readfirstlane(Tg.kto) * (size_t)B.TS;
    const uint8_t* vs = B.vov + (size_t)__builtin_amdgcn_readfirstlane(Tg.vto) * (size_t)B.TS;
    load_payload(ks, ks + SLOT_CD, lane, R.k.pay);
    load_payload(vs, vs + SLOT_CD, lane, R.v.pay);
  } else {
    // uniform 64-bit base + 32-bit byte offset per lane (one add per array; a head's arrays stay below 4 GiB, checked on the host)
    const u32 so = (u32)tile * TILE_SM + 16u * (u32)lane, co = (u32)tile * TILE_CD + 4u * (u32)lane;
    R.k.pay.s0 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(B.ksm + so));
    R.k.pay.s1 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(B.ksm + so + 1024u));
    R.v.pay.s0 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(B.vsm + so));
    R.v.pay.s1 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(B.vsm + so + 1024u));
    R.k.pay.c0 = __builtin_nontemporal_load(reinterpret_cast<const u32*>(B.kcd + co));
    R.k.pay.c1 = __builtin_nontemporal_load(reinterpret_cast<const u32*>(B.kcd + co + 256u));
    R.k.pay.c2 = __builtin_nontemporal_load(reinterpret_cast<const u32*>(B.kcd + co + 512u));
    R.v.pay.c0 = __builtin_nontemporal_load(reinterpret_cast<const u32*>(B.vcd + co));
    R.v.pay.c1 = __builtin_nontemporal_load(reinterpret_cast<const u32*>(B.vcd + co + 256u));
    R.v.pay.c2 = __builtin_nontemporal_load(reinterpret_cast<const u32*>(B.vcd + co + 512u));
  }
}
// the lane's escape position from the tag words, and the 8 escape bytes from there on
template <bool PAGED>
__device__ __forceinline__ void load_tile_escapes(const Bases& B, int lane, const TagRegs& Tg, TileRegs& R) {
  const int q = lane >> 4;
  // escape bytes per line of K (low half) and V (high half): one scan for both
  const u32 rb = (u32)esc_bytes(Tg.kfl) | ((u32)esc_bytes(Tg.vfl) << 16);
  const u32 excl = row_scan16(rb) - rb;
  // What the consumer needs of the tag words and tile offsets is computed here, into registers of the tile: the tag registers are
  // then free for the next tags, and nothing has to be copied out of a register that a load is still writing.
  R.k.f = __builtin_amdgcn_ubfe(Tg.kfl, 8 * q, 8); R.v.f = __builtin_amdgcn_ubfe(Tg.vfl, 8 * q, 8);
  R.k.pos0 = (excl & 0xFFFFu) + (u32)esc_prefix(Tg.kfl, 8 * q);
  R.v.pos0 = (excl >> 16) + (u32)esc_prefix(Tg.vfl, 8 * q);
  if (PAGED) {      // the 8-byte window stays inside the slot: a lane whose escape bytes start in the slot's last 7 bytes takes the slow look-up
    const u32 lim = (u32)(B.TS - SLOT_OV - 8);      // TS >= SLOT_OV + 16 (checked on the host)
    R.k.e = load_u32x2_unaligned(esc_of_tile<PAGED>(B.kov, __builtin_amdgcn_readfirstlane(Tg.kto), B.TS) + min(R.k.pos0, lim));
    R.v.e = load_u32x2_unaligned(esc_of_tile<PAGED>(B.vov, __builtin_amdgcn_readfirstlane(Tg.vto), B.TS) + min(R.v.pos0, lim));
  } else {      // stream base (uniform) + 32-bit offset (tile offset + position in the tile)
    R.k.pos0 += Tg.kto; R.v.pos0 += Tg.vto;
    R.k.e = load_u32x2_unaligned(B.kov + R.k.pos0);
    R.v.e = load_u32x2_unaligned(B.vov + R.v.pos0);
  }
}
template <bool PAGED>
__device__ __forceinline__ void load_tile(const Bases& B, int tile, int lane, const TagRegs& Tg, TileRegs& R) {
  load_tile_payload<PAGED>(B, tile, lane, Tg, R);
  load_tile_escapes<PAGED>(B, lane, Tg, R);
}

// ---------------------------------------------------------------------------------------------------- one tile pair
struct WaveState { f32x4 acc[8]; float m_run, mu_run, l_run; };     // acc[i][r] = O[head a][group 4q+r, element i]; m in raw score units

// The x words of the lane's four units.  Common case: 4-bit groups only -> one v_perm + four table reads.  A wave with a raw
// group somewhere (most tiles, few lanes) patches those units from the prefetched bytes.  A lane with two or more raw groups
// (its bytes may not fit the 8 prefetched ones) re-reads memory: only the SLOW instantiation contains those loads, so the
// common instantiation has no memory access between the prefetch and the products.
// bw[u]: the exponent-base words of unit u's tier, read from the block's LDS table: one table row per (tier, group), so the tier
// select costs an address bit instead of four conditional moves per unit.
// lim (SLOW only): last offset from esc_tile at which an 8-byte load may start (paged pool: the slot's end - 8; a stream: no limit).
template <int KIND, bool SLOW>
__device__ __forceinline__ void unit_x_words(const KindRegs& R, const AttnLds& L, const uint8_t* __restrict__ esc_tile, u32 lim, int a, int q,
                                             u32x4* __restrict__ x, u32x4* __restrict__ bw) {
  const u32 tag8 = R.f;
  const u32 eb4 = __builtin_amdgcn_perm(R.e[1], R.e[0], L.sel[tag8]);
  const u32x4* tab = KIND == KIND_K ? &L.bwk[0][4 * q] : &L.bwv[0][a];      // row of unit 0 at tier 0; tier 1 is NG rows further
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    x[u] = L.xlut[(eb4 >> (8 * u)) & 0xFFu];
    bw[u] = tab[(KIND == KIND_K ? u : 0) + NG * ((tag8 >> (2 * u)) & 1u)];
  }
  if (__builtin_amdgcn_ballot_w64((tag8 & 0xAAu) != 0u || (SLOW && R.pos0 > lim))) {
    const u64 e64 = (u64)R.e[0] | ((u64)R.e[1] << 32);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (((tag8 >> (2 * u)) & 3u) == 3u) {          // offset = number of 4-bit groups below (a raw one below is handled next)
        const u64 v = e64 >> (8 * __popc(tag8 & (0x55u & ((1u << (2 * u)) - 1u))));
        x[u] = raw_x_words((u32)v, (u32)(v >> 32), bw[u]);
      }
    }
    if (SLOW && (__popc(tag8 & 0xAAu) >= 2 || R.pos0 > lim)) {
      u32 off = 0u;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const u32 t = (tag8 >> (2 * u)) & 3u;
        if (t) {
          const u32 at = R.pos0 + off, from = min(at, lim);      // bytes past the limit are not this unit's: load lower, shift down
          const u64 v = load_u64_unaligned(esc_tile + from) >> (8u * (at - from));
          // The loaded bytes are waited for here, in the block that issues the load: their two users below sit in separate divergent
          // blocks, and a load that is still pending on the path past both makes the compiler wait for every load in flight wherever
          // its register is reused, on the common path as well.
          u32 vlo = (u32)v, vhi = (u32)(v >> 32);
          asm volatile("" : "+v"(vlo), "+v"(vhi));
          x[u] = t == 1u ? L.xlut[vlo & 0xFFu] : raw_x_words(vlo, vhi, bw[u]);
        }
        off += (u32)tag_size(t);
      }
    }
  }
}

// PARTIAL: the tile is the last one of the sequence and only partly filled (rows >= S are masked out).  It is a template
// parameter, not a run-time branch, so that no branch separates the score MFMAs from the first read of their result.
template <bool PAGED, bool PARTIAL>
__device__ __forceinline__ void consume(const TileRegs& R, WaveState& st, const AttnLds& L, const Bases& B,
                                        u32 kto, u32 vto, int tile, int S, float scale_log2e, int a, int q,
                                        const u32x4 (&qf)[4]) {
  // A tile needs the SLOW look-up of its escape words when some lane holds two or more raw groups (about 1 tile in 100 at 0.3 % raw
  // groups).  The choice is one wave-uniform branch around the look-ups only, ahead of all the matrix products of the tile.
  u32x4 xk[4], xv[4], bk[4], bv[4];
  const u32 kr = R.k.f & 0xAAu, vr = R.v.f & 0xAAu;
  const u32 lim = PAGED ? (u32)(B.TS - SLOT_OV - 8) : 0xFFFFFFFFu;      // paged pool: the 8 prefetched bytes were taken from no further than this
  bool slow = ((kr & (kr - 1u)) | (vr & (vr - 1u))) != 0u;
  if (PAGED) slow |= max(R.k.pos0, R.v.pos0) > lim;      // (also lanes without escape bytes: a position that far into a slot is rare)
  const bool any_slow = __builtin_amdgcn_ballot_w64(slow) != 0;
  if (__builtin_expect(any_slow, 0)) {
    unit_x_words<KIND_K, true>(R.k, L, PAGED ? esc_of_tile<PAGED>(B.kov, kto, B.TS) : B.kov, lim, a, q, xk, bk);
    if (!WAVES12) unit_x_words<KIND_V, true>(R.v, L, PAGED ? esc_of_tile<PAGED>(B.vov, vto, B.TS) : B.vov, lim, a, q, xv, bv);
  } else {
    unit_x_words<KIND_K, false>(R.k, L, nullptr, lim, a, q, xk, bk);
    if (!WAVES12) unit_x_words<KIND_V, false>(R.v, L, nullptr, lim, a, q, xv, bv);
  }
  // ---- scores: S[tok 4q+r][head a]
  f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    u32 slo, shi, w[4];
    unit_sm(R.k.pay, u, slo, shi);
    decode_unit_x(slo, shi, unit_code_word(R.k.pay.c0, R.k.pay.c1, R.k.pay.c2, u), xk[u], bk[u], w);
    const u32x4 av = {w[0], w[1], w[2], w[3]};
    const u32x4 qu = WAVES12 ? L.qw[a][4 * q + u] : qf[u];
    sacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, qu), sacc, 0, 0, 0);
  }
  if (WAVES12) {      // measurement build: the V side's look-ups only now, when the K side's registers are free
    if (__builtin_expect(any_slow, 0)) unit_x_words<KIND_V, true>(R.v, L, PAGED ? esc_of_tile<PAGED>(B.vov, vto, B.TS) : B.vov, lim, a, q, xv, bv);
    else unit_x_words<KIND_V, false>(R.v, L, nullptr, lim, a, q, xv, bv);
  }
  // ---- online softmax per head a over the tile's 16 tokens (4 in this lane, 4 quads); exp2(score * scale*log2e - mu)
  const int tok0 = tile * T + 4 * q;
  if (PARTIAL) {
#pragma unroll
    for (int r = 0; r < 4; ++r) sacc[r] = tok0 + r >= S ? -INFINITY : sacc[r];
  }
  const float tmax = quad_rows_max(fmaxf(fmaxf(sacc[0], sacc[1]), fmaxf(sacc[2], sacc[3])));
  if (__builtin_amdgcn_ballot_w64(tmax > st.m_run)) {             // the running maximum of some head grows (rare after the first tiles)
    const float mn = fmaxf(st.m_run, tmax), mu = mn == -INFINITY ? 0.f : mn * scale_log2e;
    const float alpha = __builtin_amdgcn_exp2f(st.m_run == -INFINITY ? -INFINITY : st.mu_run - mu);
    st.l_run *= alpha;
#pragma unroll
    for (int i = 0; i < 8; ++i) st.acc[i] *= alpha;
    st.m_run = mn; st.mu_run = mu;
  }
  float p[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[r], scale_log2e, -st.mu_run));
  st.l_run += (p[0] + p[1]) + (p[2] + p[3]);
  const u32x2 pw = {pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3])};
  const s16x4 pb = __builtin_bit_cast(s16x4, pw);
  // ---- values: decode the lane's 4 tokens of group a, regroup as token pairs per element, accumulate O^T
  u32 W[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    u32 slo, shi;
    unit_sm(R.v.pay, u, slo, shi);
    decode_unit_x(slo, shi, unit_code_word(R.v.pay.c0, R.v.pay.c1, R.v.pay.c2, u), xv[u], bv[u], W[u]);
  }
  if (PARTIAL) {                // rows beyond the sequence must not reach the product
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) W[u][pp] = tok0 + u >= S ? 0u : W[u][pp];
  }
#pragma unroll
  for (int pp = 0; pp < 4; ++pp) {
    const u32x2 lo = {__builtin_amdgcn_perm(W[1][pp], W[0][pp], 0x05040100u), __builtin_amdgcn_perm(W[3][pp], W[2][pp], 0x05040100u)};
    const u32x2 hi = {__builtin_amdgcn_perm(W[1][pp], W[0][pp], 0x07060302u), __builtin_amdgcn_perm(W[3][pp], W[2][pp], 0x07060302u)};
    st.acc[pp] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, lo), pb, st.acc[pp], 0, 0, 0);
    st.acc[pp + 4] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, hi), pb, st.acc[pp + 4], 0, 0, 0);
  }
}

// Next tile for a wave from the block's counter in LDS (lane 0's value counts).  The caller makes it uniform only when it needs it,
// one tile later, so that no wave waits for the LDS atomic.  Indices past the block's range come back as NO_TILE.
constexpr int NO_TILE = 0x3FFFFFFF;
__device__ __forceinline__ int take_tile(int* ctr, int hi, int lane) {
  int v = 0;
  if (lane == 0) { v = atomicAdd(ctr, 1); v = v < hi ? v : NO_TILE; }
  return v;
}
__device__ __forceinline__ int uniform_tile(int v) { return __builtin_amdgcn_readfirstlane(v); }

// ---------------------------------------------------------------------------------------------------- rows shared out by length
// Rows of a batch differ in length, and the host does not know by how much.  With the same number of splits for every row the launch lasts
// as long as a split of the longest row, while the blocks of short rows are mostly start and merge.  Here every block of the launch reads
// the B lengths and derives, in the same arithmetic and so with the same result, how many splits each row gets, and with them its own row, kv
// head and split:
//   * nearly equal rows (within 1/32 of the first one): nsplit splits per row in batch order, as without a plan, or as many as fill one round.
//   * one round: the launch uses no more blocks than are resident at once (two four-wave blocks or one eight-wave block per CU), rows get
//     splits of about c tiles, c the smallest size for which sum ceil(tiles / c) fits (found to 1/120 of c).  Blocks beyond have nothing to do.
//   * several rounds, where half a split per row, which rounding costs, is more than starting and merging blocks again and the rows do not differ
//     much, where one round would leave the longest row in pieces far above the mean, or in splits that the paged kernel's tile table does not hold: nsplit
//     splits per row, longest row first (blocks start in index order, so that the short rows fill the end of the launch).  The splits' sizes differ
//     from row to row, which keeps the rounds from starting and ending in step.  Where that would still leave the longest row in pieces far above the mean: splits
//     of about c tiles, c the smallest size for which they fit the launch's nsplit * B units, the longest first.
// The lines: a four-wave block takes about 0.5 us per tile and a round costs some 20 us of starts and merges.  16 sequences of 1000..16000
// tokens (rounding costs 17 tiles): 91 us in one round, 102 in four.  Where the rows differ, splits of many sizes meet
// on the CUs and even that out, if they are paired by size (plan_rows): paged, 8 kv heads, several rounds / one, us: 16 rows of 4096..65536 tokens (68
// tiles) 284 / 270, 32 of 500..20000 182 / 166, 24 of 2000..30000 207 / 190, 20 of 10000..40000 262 / 245.
// Measured with warm caches, 4 query heads per kv head, against equal split counts in batch order: paged, 8 sequences of 200..3000 tokens x 8
// kv heads: 27.0 -> 20.6 us, 16 of 500..6000: 71 -> 44; slot cache, 4 rows of 2000..32000: 47.4 -> 37.4, 12 of 300..8000: 53.5 -> 32.2,
// 32 of 300..6000: 68 -> 61.
// What the look at the rows costs where they turn out equal (4 rows of 32000..32768): 63.8 -> 64.0.  It is in every block's start, so it
// is kept to two trips to memory, which a block without a plan makes too, and some 300 instructions: an earlier form, which went
// through LDS, read the lengths of all B * n_kv heads in a loop and compared each row with each, took 384 us instead of 142 for 256 rows of
// 500 tokens x 16 kv heads and 64.5 for the 4 rows above.
constexpr int PLAN_ROWS = 256;           // larger batches take nsplit splits per row in batch order
constexpr float ONE_ROUND_LOSS = 48.f;   // tiles of a four-wave block
// Rows whose longest has this much over the mean go into one round also where rounding costs more.  us, slot cache / paged, several rounds -> one: 40 rows
// of 4500..7500 tokens x 8 kv heads (1.24) 144 -> 139 / 143 -> 147, 40 of 3500..8500 (1.41) 150 -> 135 / 143 -> 143, 20 of 14000..26000 (1.28) 220 -> 200 / 228 -> 204;
// but 40 of 5000..7000 (1.16) 151 -> 142 / 144 -> 150.
constexpr float ONE_ROUND_MIXED = 1.2f;
// ... if the size found is no more than this much over the mean share of a block, or ONE_ROUND_LOSS tiles above it: where there is hardly more than a unit for
// each row, the short rows take them and leave the long one in pieces that the launch waits for.  Paged, 8 kv heads, one round / several: 61 rows of 2000 tokens and
// one of 16000 (2.5 of the mean) 126 / 109 us, slot cache 116 / 102, 56 of 500..6000 (2.2) 90 / 80; 48 of 100..8000 (1.7) 111 / 116, 40 of 300..8500 (1.6) 75 / 86;
// 50 of 500 and one of 20000 (2.0, 44 tiles) 41 / 45.
constexpr float ONE_ROUND_SIZE = 1.8f;
// In several rounds the rows get splits of one size instead of nsplit each where a split of the longest would be this much over the mean share of a
// block.  us, nsplit each / one size, slot cache, two splits a row on average: 63 rows of 2000 tokens and one of 16000 x 8 kv heads (3.6) 162 / 101, 200 of 3000 and one
// of 30000 x 2 (6.1) 289 / 101, 64 of 200..8000 (1.9) 89 / 86; 56 of 500..6000 (1.5) 78 / 82; paged, 128 of 100..4000 x 4 (1.7) 70 / 75.
constexpr float SIZED_SPLIT = 1.75f;
// Smaller splits cost more in the merge than they gain: 30 sequences of up to 3000 tokens, one kv head with 16 query heads: 31.4 us
// with at least 4 tiles, 27.4 with 12, 30.1 with 20; eight sequences of up to 3000 tokens, 8 kv heads: 21.6, 21.8, 24.5.
constexpr float MIN_SPLIT_TILES = 12.f;  // of a four-wave block; half as many for an eight-wave block
// Splits of about this many tiles and up are ordered by size (plan_rows).  us, slot cache, 8 kv heads, by kind / by size; up to two units a row: 30 rows of 300 tokens
// beside one of 6000 (19 tiles) 19.1 / 21.1, 32 of 300..4000 33.2 / 32.6 (a line at 18 tiles: 34.7), 32 of 200..3000 (61) 37.2 / 35.7.  More units a
// row: 28 rows of 100..2600 (47) 31.0 / 32.1, 60 of 100..2600 x 4 heads (40) 33.5 / 36.0; from 60 tiles to 120 the two are within 1 us; 16 of
// 3000..30000 (290) 134.8 / 131, paged 142.6 / 135.6.
constexpr int SORTED_SPLIT_TILES = 28;
constexpr int SORTED_ROW_SPLITS = 2;
constexpr int LONG_SPLIT_TILES = 96;
// Two four-wave blocks share a CU, a wave of each on every SIMD, and the arbiter prefers the older one: of 16 paged rows of up to 64K tokens the
// blocks of the launch's earlier half were through after 227 us, the later half's after 287, 60 of them with half the CU's waves.  Two of the later block's
// waves go first instead, so that each block is ahead on two SIMDs (its waves share its tiles).  us, 8 kv heads: paged, 16 rows of 4096..65536 tokens
// 277 -> 270, 16 of 31000 240 -> 232; slot cache, 24 of 4000..12000 73.3 -> 69.9, 30 rows of 1000..32000 x 4 heads 62 -> 58.
//   * Only where the launch is one round (RowPlan::first): of several, bit 8 of a block's index does not tell which of two came first, and a split that
//     others put back ends later still: 40 rows of 6000 in two rounds 146 us, 179 with priorities, 40 of 5000..7000 149 and 173.
//   * Not beside a split of more than twice the length, which the CU then waits for: 61 rows of 2000 tokens and one of 16000 116 us, 126 with priorities;
//     50 of 500 and one of 20000 40.8 and 42.5.  The other block is at most as long as the plan's size of a split.
//   * Splits of a dozen tiles gain nothing: with a line at 12 tiles all within 1 us of 28; at 60, 32 rows of 300..4000 32.6 -> 35.4.
constexpr int PRIO_TILES = 28;
constexpr float PRIO_SHARE = 0.5f;
struct RowPlan { int b, S, kvh, idx, ns, off, slot; bool first; };      // idx: the block's place among the ns blocks of (row, kv head); off: splits of the rows before; first: see PRIO_TILES
__device__ __forceinline__ int plan_splits(int tiles, float c, float rc) {      // about ceil(tiles / c), the same wherever it is asked; no row (tiles < 0): none
  return tiles < 0 ? 0 : min(max((int)(((float)tiles + (c - 1.f)) * rc), 1), MAX_SLOTS);
}
// Every wave works the plan out by itself, without LDS or a barrier: lane l holds the rows l, l + 64, ..., one register each; counts are
// ballots, sums DPP, a row's place among many others is found by bisection.  false: no unit left for this block.
// K: registers of rows, B <= 64 K (a register without rows only holds lanes that are not there).
template <bool PAGED, int NW, int K>
__device__ __forceinline__ bool plan_rows(const AttnArgs& A, int lane, RowPlan& R) {
  const int B = A.B, nsplit = A.nsplit, block = (int)blockIdx.x;
  const auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const auto row = [&](int k) { return min(lane + 64 * k, B - 1); };
  // The block's place if the rows turn out equal follows from its index: slot and length of that place are loaded along with the
  // rows', so that the chain up to the block's own length has the loads of a launch without a plan.
  const int bh = uniform(div_below_2_21(block, nsplit)), b_eq = uniform(div_below_2_21(bh, A.n_kv)), kvh_eq = bh - b_eq * A.n_kv;
  const int* slots = A.slot ? A.slot : A.sl;      // (no load under a branch: without a slot map, B lengths or more are there to be read)
  int slot[K], tiles[K], slot_eq = 0;
  if (!PAGED) {
    slot_eq = slots[b_eq];
#pragma unroll
    for (int k = 0; k < K; ++k) slot[k] = slots[row(k)];
    if (!A.slot) {
      slot_eq = b_eq;
#pragma unroll
      for (int k = 0; k < K; ++k) slot[k] = row(k);
    }
  }
  const auto length = [&](int b, int s, int head) { return A.sl[PAGED ? b : max(s, 0) * A.n_kv + head]; };
  const int len_eq = length(b_eq, slot_eq, kvh_eq);
#pragma unroll
  for (int k = 0; k < K; ++k) tiles[k] = length(row(k), slot[k], 0);      // the splits go by the length of kv head 0
#pragma unroll
  for (int k = 0; k < K; ++k) tiles[k] = !PAGED && slot[k] < 0 ? 0 : (min(max(tiles[k], 0), 1 << 28) + T - 1) / T;      // (past the end: the last row again)
  bool differs = false;
  const int t0 = uniform(tiles[0]);
#pragma unroll
  for (int k = 0; k < K; ++k) differs |= 32 * abs(tiles[k] - t0) > t0;
  const bool equal = __builtin_amdgcn_ballot_w64(differs) == 0, resident = nsplit * B <= A.plan;      // equal: within 1/32 of the first row
  const auto stay = [&]() {      // at the place of equal rows
    R.b = b_eq; R.kvh = kvh_eq; R.idx = block - bh * nsplit; R.ns = nsplit; R.off = b_eq * nsplit; R.slot = slot_eq; R.S = max(len_eq, 0); R.first = resident;
    return true;
  };
  if (equal && resident) return stay();
  R.first = false;
  float total = 0.f, longest = 0.f, shortest = -INFINITY;      // (shortest: negated)
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const bool there = lane + 64 * k < B;
    const float t = (float)tiles[k];
    total += there ? t : 0.f; longest = fmaxf(longest, t); shortest = fmaxf(shortest, -t);
    tiles[k] = there ? tiles[k] : -1;
  }
  total = wave_sum(total);
  const int units = min(nsplit * B, A.plan), u = uniform(div_below_2_21(block, A.n_kv));     // a unit is a split for every kv head: n_kv blocks
  const float fu = (float)units;
  int ns = nsplit, b = 0, off = 0, w = -1;      // w: the block's place among the ns blocks of each of the row's kv heads, where that is not block - off * n_kv
  if (equal) {
    // batch order, with nsplit splits per row, or as many as make one round where that loses less than several rounds, or where the last
    // of several rounds would be much emptier (24 rows of 12000 tokens x 8 kv heads, 3 splits: 576 blocks 171 us, 2 splits 152)
    if (!resident && nsplit > 1 && units >= B) {
      const int n1 = uniform(div_below_2_21(units, B)), rounds = uniform(div_below_2_21(nsplit * B + units - 1, units));
      const float loss = wave_max(longest) * __builtin_amdgcn_rcpf((float)n1) - total * __builtin_amdgcn_rcpf(fu);
      if (10 * nsplit < 9 * rounds * n1 || __builtin_amdgcn_ballot_w64(loss > ONE_ROUND_LOSS) == 0) ns = n1;
    }
    if (ns == nsplit) return stay();
    b = uniform(div_below_2_21(u, ns)); off = b * ns; R.first = true;
    if (b >= B) return false;
  } else {
    const auto holds = [](bool v) { return __builtin_amdgcn_ballot_w64(v) != 0; };      // (of values that are the same in all lanes)
    // half a split per row goes to rounding: total / units * B / (2 units) tiles on every block
    const bool can = nsplit > 1 && units >= B;
    bool mixed = false, try_one = can && (resident || holds(total * (float)B <= ONE_ROUND_LOSS * 2.f * fu * fu));
    if (K == 1 && __builtin_expect(can && !try_one, 0)) try_one = mixed = holds(wave_max(longest) * (float)B > ONE_ROUND_MIXED * total);
    float c_best = 0.f;
    const auto find_size = [&](int use) {      // c_best: the smallest size whose splits fit `use` units; 0 if there is none
      // sixteen sizes from the mean to three times that, then sixteen between the first that fits and the one before it; lane (j, r) =
      // (lane & 15, lane >> 4) tries size j over the rows r, r + 4, ...
      const float c_min = fmaxf(floorf(total * __builtin_amdgcn_rcpf((float)use)) + 1.f, NW == 4 ? MIN_SPLIT_TILES : 0.5f * MIN_SPLIT_TILES), step = c_min * (2.f / 15.f);
      float lo = c_min, width = step;
#pragma unroll 1
      for (int pass = 0; pass < 2; ++pass) {
        const float c = lo + width * (float)(lane & 15), rc = __builtin_amdgcn_rcpf(c);
        float n = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) {
#pragma unroll 1
          for (int i = 0; i < (K > 1 ? 64 : B); i += 16)      // (lanes without a row take no splits)
#pragma unroll
            for (int j = 0; j < 16; j += 4) n += (float)plan_splits(__builtin_amdgcn_ds_bpermute(4 * (i + j + (lane >> 4)), tiles[k]), c, rc);
        }
        n = quad_rows_sum(n);
        const u64 fits = __builtin_amdgcn_ballot_w64(n <= (float)use) & 0xFFFFull;
        if (fits) c_best = __uint_as_float((u32)__builtin_amdgcn_readlane((int)__float_as_uint(c), __builtin_ctzll(fits)));
        if (K > 1 && uniform((int)c_best) == 0) break;      // (with K 1 the second look costs less than the branch: it tries what did not fit again)
        lo = fmaxf(c_best - step, c_min); width = step * (1.f / 16.f);
      }
    };
    if (try_one) {
      find_size(units);
      if (PAGED && !resident) c_best = c_best <= (float)MAX_CHUNK ? c_best : 0.f;
      if (__builtin_expect(mixed, 0)) {
        const float mean = total * __builtin_amdgcn_rcpf(fu);
        c_best = c_best <= fmaxf(ONE_ROUND_SIZE * mean, mean + ONE_ROUND_LOSS) ? c_best : 0.f;
      }
    }
    const int c_int = uniform((int)c_best);
    const bool one_round = c_int != 0;
    b = -1;
    const auto long_split = [&](int row_tiles) { return holds((float)row_tiles >= PRIO_SHARE * c_best * (float)ns); };
    if (__builtin_expect(one_round && (K > 1 || NW != 4 || c_int < (units <= SORTED_ROW_SPLITS * B ? SORTED_SPLIT_TILES : LONG_SPLIT_TILES)), 1)) {
      const float rc = __builtin_amdgcn_rcpf(c_best);
      // Short splits, and more rows than a wave has lanes: the rows of several splits, whose blocks are all long and are waited for by a merge, come first,
      // then the others, either in batch order (100 rows of 100..4000 x 4 kv heads 70.5 us, all longest first 77).  The counts of the two
      // kinds run in the halves of one word.
      u32 n[K], end[K], sum = 0u;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        n[k] = (u32)plan_splits(tiles[k], c_best, rc);
        n[k] = n[k] > 1u ? n[k] : n[k] << 16;
        const u32 x = row_scan16(n[k]), r0 = __builtin_amdgcn_readlane(x, 15), r1 = __builtin_amdgcn_readlane(x, 31), r2 = __builtin_amdgcn_readlane(x, 47);
        end[k] = sum + x + (lane >= 16 ? r0 : 0u) + (lane >= 32 ? r1 : 0u) + (lane >= 48 ? r2 : 0u);
        sum = (u32)__builtin_amdgcn_readlane((int)end[k], 63);
      }
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const bool several = n[k] < 65536u;
        const int mine = several ? (int)n[k] : (int)(n[k] >> 16), to = several ? (int)(end[k] & 65535u) : (int)((end[k] >> 16) + (sum & 65535u));
        const u64 own = __builtin_amdgcn_ballot_w64(u >= to - mine && u < to);
        if (own != 0) {
          const int l = __builtin_ctzll(own);
          b = 64 * k + l; ns = __builtin_amdgcn_readlane(mine, l); off = __builtin_amdgcn_readlane(to, l) - ns;
          R.first = long_split(__builtin_amdgcn_readlane(tiles[k], l));
          break;
        }
      }
    } else {
      bool sized = can && !one_round && holds(wave_max(longest) > SIZED_SPLIT * (float)nsplit * total * __builtin_amdgcn_rcpf(fu));
      if (sized) {      // (with two splits a row and up, three times the mean always fits)
        find_size(nsplit * B);
        sized = uniform((int)c_best) != 0;
      }
      const float rc = __builtin_amdgcn_rcpf(c_best);
      if (K == 1) {
        // The longest splits first, or the longest row where each has nsplit.  A lane adds up the splits of the rows ahead of its own.
        // One round: all blocks start together, two four-wave blocks to a CU, the later half of the launch beside the earlier one, and in the later half the
        // shortest go first, so that every CU gets about the same.
        // (With the order turning at the 256th block, where the second ones come, 300 to 400 blocks take the same to 1 us.)
        // By kind, as above -> by size, us, 8 kv heads: 32 rows of 300..6000 tokens 61.6 -> 55.5, 48 of 100..8000 79.9 -> 65.1, 28 of 300..6000
        // 60.2 -> 55.7, 32 of 100..2000 29.6 -> 27.9, 20 of 100..16000 55.8 -> 54.2; with four classes of size 62.3 for the first.
        const bool by_size = one_round || sized;
        const int n = by_size ? min(plan_splits(tiles[0], c_best, rc), 1023) : tiles[0] < 0 ? 0 : nsplit, mask = by_size ? 1023 : 0, add = by_size ? 0 : nsplit;
        const int key = by_size && tiles[0] >= 0 ? min((int)((float)tiles[0] * __builtin_amdgcn_rcpf((float)n) * rc * 16383.f), 32767) << 16 | (63 - lane) << 10 | n
                                                 : tiles[0] * 64 + 63 - lane;      // (below zero: not there)
        int before = 0;
#pragma unroll 1
        for (int i = 0; i < B; i += 8)
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            const int other = __builtin_amdgcn_readlane(key, i + r);
            before += other > key ? (other & mask) + add : 0;
          }
        const int used = (one_round ? units : nsplit * B) * A.n_kv, half = one_round ? (units >> 1) * A.n_kv : used;
        if (block >= used) return false;
        const int v = block < half ? block : used - 1 - (block - half), uv = uniform(div_below_2_21(v, A.n_kv));      // the block's place in that order
        const u64 own = __builtin_amdgcn_ballot_w64(uv >= before && uv < before + n);
        if (own == 0) return false;
        b = __builtin_ctzll(own); ns = __builtin_amdgcn_readlane(n, b); off = __builtin_amdgcn_readlane(before, b);
        R.first = one_round && long_split(__builtin_amdgcn_readlane(tiles[0], b));
        // a head's splits in the order of the blocks' indexes also where that runs backwards (see merge_heads: a merger waits for blocks that start before it)
        const int row0 = off * A.n_kv;
        w = block < half ? v - row0 : max(row0, half) + ns * A.n_kv - 1 - v;
      } else {
        // Several rounds of more rows than a wave has lanes, longest row first: the splits of the rows longer than m tiles become fewer as m grows, and
        // the block's row is where they pass its place.
        const auto splits_above = [&](int m) {
          int n = 0;
          if (sized) {
#pragma unroll
            for (int k = 0; k < K; ++k) n += tiles[k] > m ? plan_splits(tiles[k], c_best, rc) : 0;
            return uniform((int)wave_sum((float)n));
          }
#pragma unroll
          for (int k = 0; k < K; ++k) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(tiles[k] > m));
          return n * nsplit;
        };
        int below = uniform((int)-wave_max(shortest)) - 1, own = uniform((int)wave_max(longest)), ahead = 0;
        if (splits_above(below) <= u) return false;
#pragma unroll 1
        while (own - below > 1) {
          const int mid = (own + below) >> 1, n = splits_above(mid);
          if (n <= u) { own = mid; ahead = n; } else below = mid;
          if (n == u) break;
        }
        if (ahead == u) {      // the next row of up to `own` tiles
          float t = -1.f;
#pragma unroll
          for (int k = 0; k < K; ++k) t = fmaxf(t, tiles[k] <= own ? (float)tiles[k] : -1.f);
          own = uniform((int)wave_max(t));
        }
        if (sized) ns = uniform(plan_splits(own, c_best, rc));
        int rank = uniform(div_below_2_21(u - ahead, ns));      // the block's row is the rank-th, in batch order, of those of this length
        off = ahead + rank * ns;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const u64 m = __builtin_amdgcn_ballot_w64(tiles[k] == own);
          const int n = __builtin_popcountll(m);
          if (rank < n) {
            const int before = __builtin_amdgcn_mbcnt_hi((u32)(m >> 32), __builtin_amdgcn_mbcnt_lo((u32)m, 0u));
            b = 64 * k + __builtin_ctzll(__builtin_amdgcn_ballot_w64(tiles[k] == own && before == rank));
            break;
          }
          rank -= n;
        }
      }
    }
    if (b < 0) return false;
  }
  if (w < 0) w = block - off * A.n_kv;
  R.b = b; R.ns = ns; R.off = off; R.kvh = uniform(div_below_2_21(w, ns)); R.idx = w - R.kvh * ns;
  R.slot = 0;
  if (!PAGED) {
#pragma unroll
    for (int k = 0; k < K; ++k) if (b >> 6 == k) R.slot = __builtin_amdgcn_readlane(slot[k], b & 63);
  }
  R.S = max(length(b, R.slot, R.kvh), 0);      // (the line is at hand from the look at the rows)
  return true;
}
template <bool PAGED, int NW>
__device__ __forceinline__ bool plan_block(const AttnArgs& A, int lane, RowPlan& R) {
  return __builtin_expect(A.B <= 64, 1) ? plan_rows<PAGED, NW, 1>(A, lane, R) : plan_rows<PAGED, NW, PLAN_ROWS / 64>(A, lane, R);
}

// ---------------------------------------------------------------------------------------------------- main kernel
// NW = waves per block: 4 (two blocks per CU) or 8 (one block per CU: half as many partials to merge for the same occupancy)
// HOST_LEN: the compressed length of every addressed head is the kernel argument S_all (not read from memory)
template <bool PAGED, int NW, bool HOST_LEN>
__global__ void __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) k_attn_split(const AttnArgs A) {
  constexpr int NT = 64 * NW;
  // Raw tiles of the paged pool: a wave for every four of the block, so that a CU has two in either launch form.  Pools of raw tiles only, 8 kv heads, one / two
  // in an eight-wave block, us: 8 rows of 200..3000 tokens 48 / 31.5, 4 of 1000..9000 65 / 42, one of 30000 88 / 54.4.
  constexpr int RAWS = PAGED && NW == 8 ? 2 : 1;
  // one LDS object so that the tables the tile loop reads sit at the lowest addresses (immediate offsets of the LDS loads)
  struct BlockLds { AttnLds L; int next_tile, two_raws; int2 tile_table[PAGED ? MAX_CHUNK : 1]; MergeLds<NW, RAWS> M; };
  static_assert(offsetof(BlockLds, M.acc) % 16 == 0, "the block merge's accumulators are stored and a decoded raw tile is read 16 bytes at a time");
  __shared__ BlockLds lds;
  AttnLds& L = lds.L; MergeLds<NW, RAWS>& M = lds.M; int2* tile_table = lds.tile_table; int& next_tile = lds.next_tile;
  const int tid = threadIdx.x;
  GAAC_STAMP(0);
  // One-dimensional grid, numbered split-fastest: the splits of one kv head go round the eight XCDs (workgroups are dealt to XCDs in
  // turn) instead of all landing on one, so heads with heavier tiles load every XCD alike.
  // The start of a block is a chain of dependent loads (arguments -> slot -> lengths and stream starts -> tag words -> escape bytes),
  // each a trip to memory with nothing else to do: issue everything a level allows before the first use of any of its results.
  // Level 0: the kernel arguments, forced into scalar registers together (otherwise each is fetched where it is first used).
  if (PAGED)
    asm volatile("" ::"s"(A.q), "s"(A.sl), "s"(A.bt), "s"(A.mt), "s"(A.pool), "s"(A.raw), "s"(A.k.base3), "s"(A.k.base4), "s"(A.v.base3),
                 "s"(A.v.base4), "s"(A.nsplit), "s"(A.n_kv), "s"(A.n_q), "s"(A.G), "s"(A.NB), "s"(A.bt_stride), "s"(A.TS));
  else
    asm volatile("" ::"s"(A.q), "s"(A.slot), "s"(A.sl), "s"(A.k.sm), "s"(A.k.cd), "s"(A.k.flags), "s"(A.k.tile_off), "s"(A.k.ovf),
                 "s"(A.k.head_start), "s"(A.k.base3), "s"(A.k.base4), "s"(A.v.sm), "s"(A.v.cd), "s"(A.v.flags), "s"(A.v.tile_off),
                 "s"(A.v.ovf), "s"(A.v.head_start), "s"(A.v.base3), "s"(A.v.base4), "s"(A.kt), "s"(A.tl), "s"(A.nsplit), "s"(A.n_kv),
                 "s"(A.n_q), "s"(A.G), "s"(A.NB), "s"(A.S_pad), "s"(A.tcap));
  // Paged pool: the launch can take the place of gaac_paged_free (it pops nothing, so pushes are safe here): the grid's last block, the
  // one with the least to do, pushes the queued raw tiles back before its own work.  The wait keeps the stores' bookkeeping out of
  // the code every block runs.
  if (PAGED && A.freeq != nullptr && blockIdx.x == gridDim.x - 1) {
    for (int i = tid; i < A.n_free; i += NT) { const int r = A.freeq[i]; if (r >= 0) A.stack[atomicAdd(A.top, 1)] = r; }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  const int G = A.G;
  RowPlan R;
  if (!HOST_LEN && __builtin_expect(A.plan != 0, 0)) {
    if (!plan_block<PAGED, NW>(A, tid & 63, R)) {
      if (A.nslot > 1) {      // no unit left for this block: it only takes its part in the launch's epoch
        const u32 epoch = load_epoch(A);
        if (tid == 0) mark_arrival(A, epoch);
        if (blockIdx.x == gridDim.x - 1) {
          MarkRegs<NW> xm;
          load_marks<NW>(A, tid, xm);
          advance_epoch<NW>(A, epoch, tid, xm, &M.m[0][0], 1);
        }
      }
      return;
    }
  } else {
    const int bh = __builtin_amdgcn_readfirstlane(small_div(blockIdx.x, A.nsplit));
    R.b = __builtin_amdgcn_readfirstlane(small_div(bh, A.n_kv)); R.kvh = bh - R.b * A.n_kv; R.idx = (int)blockIdx.x - bh * A.nsplit; R.ns = A.nsplit; R.off = R.b * A.nsplit; R.S = -1; R.first = gridDim.x <= 512u;
    // (no slot map = row b attends over cache heads b*n_kv ..: one level of dependent loads less)
    R.slot = PAGED ? 0 : (A.slot ? A.slot[R.b] : R.b);
    if (!PAGED && !HOST_LEN) R.S = A.sl[max(R.slot, 0) * A.n_kv + R.kvh];
  }
  const int b = R.b, kvh = R.kvh, ns = R.ns;
  // Paged pool: the split index is rotated by the head's place in the grid: the last split of a sequence carries the raw tile that is still filling,
  // and all of them would otherwise sit on the same XCD whenever the split count is a multiple of eight, which then finishes long after the others.
  const int turn = R.idx + ((R.off * A.n_kv) >> 4) + kvh;
  const int split = PAGED ? turn - ns * __builtin_amdgcn_readfirstlane(small_div(turn, ns)) : R.idx;
  const long qh0 = (long)b * A.n_q + (long)kvh * G;
  // Level 1: the slot of the batch row; the query rows do not depend on it
  TableRegs Tr;
  if (tid < 256) tables_load_q(Tr, tid, A.q + qh0 * D, G);
  const int slot = R.slot, ch = PAGED ? kvh : (slot < 0 ? 0 : slot) * A.n_kv + kvh;
  // Level 2: everything indexed by the cache head
  int S, TLh = 0; long khs = 0, vhs = 0;
  if (PAGED) S = R.S >= 0 ? R.S : max(A.sl[b], 0);
  else {
    // lengths known to the host (a Page) come as a kernel argument: the tile range, and with it the first payload loads, then depend on
    // nothing but the arguments
    // These values are needed late (escape bytes, tail).  The index goes through a vector register the compiler knows nothing
    // about, so that the loaded values stay in vector registers until readfirstlane fetches them where they are used; a value the
    // compiler knows to be uniform is moved to a scalar register, and waited for, right where it is loaded.
    int chv = ch;
    asm volatile("" : "+v"(chv));
    khs = A.k.head_start[chv]; vhs = A.v.head_start[chv];
    TLh = (A.kt ? A.tl : A.k.head_start)[chv];      // no branch between the loads of this level
    if (HOST_LEN) S = A.S_all;
    else S = R.S;
    if (slot < 0) S = 0;
  }
  if (tid < 256) tables_load_bases(Tr, tid, A.k.base3, A.k.base4, A.v.base3, A.v.base4, ch - A.NB * __builtin_amdgcn_readfirstlane(small_div(ch, A.NB)));

  const int ntiles = (S + T - 1) / T, chunk = __builtin_amdgcn_readfirstlane(small_div(ntiles + ns - 1, ns));
  const int tlo = min(split * chunk, ntiles), thi = min(tlo + chunk, ntiles);
  const int thi_fast = PAGED ? min(thi, tlo + MAX_CHUNK) : thi;      // the pipelined loop's range: what one fill of the LDS tile table covers
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, a = lane & 15, q = lane >> 4;
  Bases B;
  TileTable TT{tile_table, tlo};
  // Waves that the split's raw tiles are shared out to, in turn.  Most splits have none or one, the filling block's: then wave 0 at most, and no further partial to merge.
  // (A second wave that looked for itself, and its partial in every merge: one row of 300 tokens x 8 kv heads 10.4 -> 11.2 us, of 900 11.9 -> 12.4, 12 of 130..460 x 4 13.1 -> 13.2.)
  int raws = 0;
  const auto count_raws = [&](bool raw, bool first) {      // (threads with a raw tile: one that has two, 512 apart, leaves both to wave 0)
    raws = RAWS > 1 ? min(__syncthreads_count(raw), RAWS) : (int)__syncthreads_or(raw);
    // whether any round of the split has two, for the merge: in LDS, as a register for it costs the tile loop (20 rows of 100..500 x 8 14.2 -> 14.05)
    if (RAWS > 1 && tid == 0 && (first || raws > 1)) lds.two_raws = raws > 1;
  };
  if (PAGED) {
    // logical tile -> block table -> mode table (paged_kernel.py:137-138), resolved once per block into LDS
    B.kov = B.vov = A.pool; B.TS = A.TS;
    B.ksm = B.kcd = B.vsm = B.vcd = nullptr; B.kfl = B.kto = B.vfl = B.vto = nullptr;
    bool raw = false;
    for (int i = tid; i < thi_fast - tlo; i += NT) {
      const long pc = (long)A.bt[(long)b * A.bt_stride + tlo + i] * (2 * A.n_kv) + 2 * kvh;
      const int2 e = {A.mt[pc], A.mt[pc + 1]};
      tile_table[i] = e;
      raw |= (e.x | e.y) < 0;
    }
    count_raws(raw, true);
  } else {
    const long rowb = (long)ch * A.S_pad, tileb = (long)ch * (A.S_pad / T);
    // (the escape streams start at head_start[ch], a loaded value: they are set where the first escape bytes are fetched, so that the
    // loads issued until then do not wait for it)
    B.ksm = A.k.sm + rowb * D; B.kcd = A.k.cd + rowb * CB; B.kfl = A.k.flags + rowb; B.kto = A.k.tile_off + tileb; B.kov = nullptr;
    B.vsm = A.v.sm + rowb * D; B.vcd = A.v.cd + rowb * CB; B.vfl = A.v.flags + rowb; B.vto = A.v.tile_off + tileb; B.vov = nullptr;
    B.TS = 0;
  }

  // Tiles are handed out dynamically: each wave starts with tiles tlo + wave and tlo + NW + wave and takes every further one from
  // a counter in LDS.  Of the two waves that share a SIMD the older one wins the issue arbitration and runs ahead; with a static
  // split it would finish long before the other, which then runs alone and cannot hide its own latencies.  Ping-pong registers
  // R0/R1; tag words are fetched one tile further ahead; indices past the end are clamped for the loads (no load sits under a
  // branch the consumer has to join) and not consumed.  A partly filled last tile of the sequence follows at the end, by the first wave without a tile of its own.
  // logical tile index i of this block -> tile tlo + i
  const int full = ntiles - ((S % T) != 0 ? 1 : 0);      // tiles with all 16 rows
  const int n_own = max(min(thi_fast, full) - tlo, 0);
  const int icl = max(n_own - 1, 0);
#define TILE(i) (tlo + (i))
  int iA = wave, iB = wave + NW;
  TileRegs R0, R1;
  // Two sets of tag registers, used in turn: a set is loaded one tile before the payload that needs it, read where that payload's
  // escape bytes are fetched, and then free.  (Paged pool: slot indices and the raw mark of the tile in R0 / R1, scalar values.)
  TagRegs Tg, TgB;
  struct TileMeta { u32 kto, vto; int raw; } m0 = {0u, 0u, 0}, m1 = {0u, 0u, 0};
  const bool any_tile = iA < n_own;
  // The wave's first tile: tag words and payload.  Without a branch where the addresses are always valid (a wave without tiles reads
  // a tile it does not consume): behind a branch the compiler can no longer count the loads in flight and turns every later wait
  // into a wait for all of them.  The escape bytes, which need the tag words and the stream start, follow after the block tables.
  if (!PAGED || any_tile) {
    const int tA = min(TILE(min(iA, icl)), max(ntiles - 1, 0));
    load_tags<PAGED>(B, TT, tA, a, Tg);
    load_tile_payload<PAGED>(B, tA, lane, Tg, R0);
  }
  if (tid == 0) next_tile = 2 * NW;
  // this launch's epoch of the fused merge: one more load of the start-up batch, its value is needed when the block is done
  const u32 epoch = load_epoch(A);
  GAAC_STAMP(6);
  if (tid < 256) tables_store(L, Tr, tid, G);
  GAAC_STAMP(7);
  if (tid < RAWS * GMAX) { M.m[NW + tid / GMAX][tid % GMAX] = -INFINITY; M.l[NW + tid / GMAX][tid % GMAX] = 0.f; }
  lds_barrier();        // block tables are ready (a barrier that does not wait for the tile loads in flight)
  GAAC_STAMP(1);
  // Q as the B operand of the score product: lane (head a, quad q), product u covers group 4q+u in word order (e, e+4);
  // exponent-base words of the lane's units
  u32x4 qf[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) qf[u] = L.qw[a][4 * q + u];

  WaveState st;
#pragma unroll
  for (int i = 0; i < 8; ++i) st.acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  st.m_run = -INFINITY; st.mu_run = 0.f; st.l_run = 0.f;

  // ---- uncompressed rows, taken by wave 0 before it joins the tile hand-out: the raw tail of the cache head (in the last split's block), or
  // the raw tiles of the paged pool among the split's tiles
  if (!PAGED && A.kt && split == ns - 1 && wave == 0) {
    const int TL = slot < 0 ? 0 : min(__builtin_amdgcn_readfirstlane(TLh), A.tcap);
    if (TL > 0) {
      u32x4 qr[4];
      raw_queries(A.q + qh0 * D, G, a, q, qr);
      RawState rs = {};
      rs.m = -INFINITY;
      raw_rows_attend(A.kt + (long)ch * A.tcap * D, A.vt + (long)ch * A.tcap * D, TL, qr, A.scale_log2e, a, q, rs);
      raw_rows_store(rs, a, q, M.m[NW], M.l[NW], M.acc[NW]);
    }
  }
  // Paged pool, wave 0, or waves 0 and 1 in turn (raws): the tiles c0 .. c1 - 1, whose entries the table holds, that have a raw side (the block that is still filling, or
  // escapes that did not fit the slot).  Raw sides are read in place, the compressed side of a half raw tile is decoded into LDS.
  const auto attend_raw_tiles = [&](int c0, int c1) {
    RawState rs;
    u32x4 qr[4];
    raw_queries(A.q + qh0 * D, G, a, q, qr);
    raw_rows_load(rs, a, q, M.m[NW + wave], M.l[NW + wave], M.acc[NW + wave]);
    u16* decoded = reinterpret_cast<u16*>(&M.acc[wave][0][0]);      // (the wave's own place in the block merge)
    int turn = wave;      // even: the next raw tile is this wave's
    const long boff = (long)(ch % A.NB) * D;
    for (int i0 = 0; i0 < c1 - c0; i0 += 64) {
      const int2 own = tile_table[min(i0 + lane, c1 - c0 - 1)];
      const bool raw = i0 + lane < c1 - c0 && (own.x | own.y) < 0;
      u64 left = __builtin_amdgcn_ballot_w64(raw);
      if (RAWS > 1 && raws > 1) {      // every other one
        const int ahead = __builtin_amdgcn_mbcnt_hi((u32)(left >> 32), __builtin_amdgcn_mbcnt_lo((u32)left, 0));
        const int next = turn + __builtin_popcountll(left);
        left = __builtin_amdgcn_ballot_w64(raw && ((turn + ahead) & 1) == 0);
        turn = next;
      }
      for (; left != 0; left &= left - 1) {
        const int l = __builtin_ctzll(left), ex = __builtin_amdgcn_readlane(own.x, l), ey = __builtin_amdgcn_readlane(own.y, l);
        const u16* krows = decoded; const u16* vrows = decoded;
        wave_lds_sync();
        if (ex < 0) krows = A.raw + (long)(~ex) * T * D;
        else {
          const uint8_t* sl = A.pool + (size_t)ex * (size_t)A.TS;
          decode_tile_rows<KIND_K>(sl, sl + SLOT_CD, reinterpret_cast<const int*>(sl + SLOT_FL), sl + SLOT_OV, A.k.base3 + boff, A.k.base4 + boff, lane, T, decoded, D);
        }
        if (ey < 0) vrows = A.raw + (long)(~ey) * T * D;
        else {
          const uint8_t* sl = A.pool + (size_t)ey * (size_t)A.TS;
          decode_tile_rows<KIND_V>(sl, sl + SLOT_CD, reinterpret_cast<const int*>(sl + SLOT_FL), sl + SLOT_OV, A.v.base3 + boff, A.v.base4 + boff, lane, T, decoded, D);
        }
        wave_lds_sync();
        raw_rows_attend(krows, vrows, min(T, S - (c0 + i0 + l) * T), qr, A.scale_log2e, a, q, rs);
      }
    }
    raw_rows_store(rs, a, q, M.m[NW + wave], M.l[NW + wave], M.acc[NW + wave]);
  };
  if (PAGED && wave < raws) attend_raw_tiles(tlo, thi_fast);

  if (!PAGED) { B.kov = A.k.ovf + __builtin_amdgcn_readfirstlane((int)khs); B.vov = A.v.ovf + __builtin_amdgcn_readfirstlane((int)vhs); }
  if (NW == 4 && R.first && n_own >= PRIO_TILES && (blockIdx.x & 256u) != 0u && wave < 2) __builtin_amdgcn_s_setprio(1);
  if (any_tile) {
    if (PAGED) m0 = TileMeta{Tg.kto, Tg.vto, Tg.raw};
    load_tile_escapes<PAGED>(B, lane, Tg, R0);
    load_tags<PAGED>(B, TT, TILE(min(iB, icl)), a, TgB);
    int vC = take_tile(&next_tile, n_own, lane);
    // The loop is entered with the loads in flight in the same order as on its back edge (tile, then the next tile's tags), so the
    // waits inside it stay waits for exactly the loads they need.
    while (true) {        // R0 = tile iA, TgB = tags of tile iB
      if (PAGED) m1 = TileMeta{TgB.kto, TgB.vto, TgB.raw};
      load_tile<PAGED>(B, TILE(min(iB, icl)), lane, TgB, R1);
      const int vD = take_tile(&next_tile, n_own, lane);
      const int iC = uniform_tile(vC);
      load_tags<PAGED>(B, TT, TILE(min(iC, icl)), a, Tg);
      if (!PAGED || !m0.raw) consume<PAGED, false>(R0, st, L, B, m0.kto, m0.vto, TILE(iA), S, A.scale_log2e, a, q, qf);
      if (iB >= n_own) break;
      if (PAGED) m0 = TileMeta{Tg.kto, Tg.vto, Tg.raw};
      load_tile<PAGED>(B, TILE(min(iC, icl)), lane, Tg, R0);
      const int vE = take_tile(&next_tile, n_own, lane);
      const int iD = uniform_tile(vD);
      load_tags<PAGED>(B, TT, TILE(min(iD, icl)), a, TgB);
      if (!PAGED || !m1.raw) consume<PAGED, false>(R1, st, L, B, m1.kto, m1.vto, TILE(iB), S, A.scale_log2e, a, q, qf);
      if (iC >= n_own) break;
      iA = iC; iB = iD; vC = vE;
    }
  }
#undef TILE
  if (NW == 4) __builtin_amdgcn_s_setprio(0);
  // arrival mark of the block for the fused merge (see merge_heads): the wave has no load in flight here
  if (A.epochs != nullptr && A.nslot > 1 && tid == 0) mark_arrival(A, epoch);
  GAAC_STAMP(2);
#ifdef GAAC_PHASE_TIMING
  if (A.dbg && lane == 0) A.dbg[((long)gridDim.x + blockIdx.x) * 8 + wave] = wall_clock64();
#endif
  // ---- what the pipelined loop left: (1) the partly filled last tile of the sequence; (2) paged pool: a split longer than the LDS tile
  // table goes on in further rounds of MAX_CHUNK tiles (table refilled, raw tiles again by the same waves).  Tiles are taken by the waves in turn, one
  // at a time without the prefetch pipeline (of the block's waves some compute while others wait for their tile; both cases are
  // rare), through ONE instantiation of the masking tile code.
  if (tlo < thi) {
    for (int c0 = tlo;;) {
      const int c1 = PAGED ? min(c0 + MAX_CHUNK, thi) : thi;
      if (PAGED && c0 != tlo) {
        __syncthreads();      // everybody is done with the previous round's entries
        bool raw = false;
        for (int i = tid; i < c1 - c0; i += NT) {
          const long pc = (long)A.bt[(long)b * A.bt_stride + c0 + i] * (2 * A.n_kv) + 2 * kvh;
          const int2 e = {A.mt[pc], A.mt[pc + 1]};
          tile_table[i] = e;
          raw |= (e.x | e.y) < 0;
        }
        count_raws(raw, false);
        TT.tlo = c0;
        if (wave < raws) attend_raw_tiles(c0, c1);
      }
      // first round: only the partial tile is left, for the first wave that has no tile of its own, if there is one (it waits for tag words,
      // then for escape bytes: behind wave 0's own tiles 1000 tokens x 8 kv heads in 16 splits took 9.6 us instead of 8.6)
      const int first = c0 == tlo ? min(n_own, NW - 1) : 0;
      for (int t = (c0 == tlo ? tlo + n_own : c0) + (wave >= first ? wave - first : wave - first + NW); t < c1; t += NW) {
        load_tags<PAGED>(B, TT, t, a, Tg);
        load_tile<PAGED>(B, t, lane, Tg, R0);
        if (!PAGED || !Tg.raw) consume<PAGED, true>(R0, st, L, B, Tg.kto, Tg.vto, t, S, A.scale_log2e, a, q, qf);
      }
      c0 = c1;
      if (c0 >= thi) break;
    }
  }
  // The accumulators are MFMA results: keep their first non-MFMA read a full MFMA latency away on every path.
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
  GAAC_STAMP(3);
  float l_run = quad_rows_sum(st.l_run);
  const float m_run = st.m_run == -INFINITY ? -INFINITY : st.mu_run;     // partial maxima are stored in the base-2 domain
  f32x4 (&acc)[8] = st.acc;

  // ---- merge the waves of the block, write the split's partial
  if (a < G) {
    if (q == 0) { M.m[wave][a] = m_run; M.l[wave][a] = l_run; }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int r = 0; r < 2; ++r)      // elements r and r + 2 are the adjacent channels 64 r + 8 i + 2 q, + 1
        *reinterpret_cast<float2*>(&M.acc[wave][a][chan_v(8 * (4 * q + r) + i)]) = float2{acc[i][r], acc[i][r + 2]};
  }
  GAAC_MSTAMP(5, wall_clock64());
  lds_barrier();      // only LDS data crosses (a full barrier would also wait for the acknowledgement of the arrival mark)
  GAAC_MSTAMP(6, wall_clock64());
  const bool fused = A.epochs != nullptr;
  const int mergers = merge_ranks(G, ns), rank = R.idx - (ns - mergers);      // the head's last blocks to start
  const long rec0 = (long)R.off * A.n_q + (long)(kvh * G) * ns;      // the group's first record
  // A wave takes 64 * C channels of a head from c0 on, a lane every 64th of them (adjacent channels of a lane would spread a wave's records over twice
  // the lines).  Latency: reads, exponentials, stores; one pass where it was two for more query heads than half the waves.  Paged, 8 sequences of 200..3000
  // tokens x 8 kv heads 23.6 -> 23.1 us with the store, 4000 tokens x 1 kv head of 16 10.1 -> 9.6.  (Without the barrier between this and the split
  // merge, which then needs LDS of its own: 64K x 4 of 6 22.3 -> 22.8.)
  const auto merge_block = [&](auto channels, auto partials, int g, int c0) {
    constexpr int C = decltype(channels)::value, P = decltype(partials)::value;
    // every LDS read up front and none under a branch: nine dependent round trips otherwise
    float mv[P], lv[P], av[P][C];
#pragma unroll
    for (int w = 0; w < P; ++w) {
      mv[w] = M.m[w][g]; lv[w] = M.l[w][g];
#pragma unroll
      for (int c = 0; c < C; ++c) av[w][c] = M.acc[w][g][c0 + 64 * c + lane];
    }
    float Mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < P; ++w) Mx = fmaxf(Mx, mv[w]);
    float Lc = 0.f, Ac[C] = {};
#pragma unroll
    for (int w = 0; w < P; ++w) {
      const bool live = mv[w] != -INFINITY;          // an empty partial's accumulator may hold anything
      const float f = live ? __builtin_amdgcn_exp2f(mv[w] - Mx) : 0.f;
      Lc += lv[w] * f;
#pragma unroll
      for (int c = 0; c < C; ++c) Ac[c] += (live ? av[w][c] : 0.f) * f;
    }
    const long pidx = rec0 + (long)g * ns + split;
    const bool lead = c0 == 0 && lane == 0;
    if (!fused) {
      if (lead) { store_partial(A.pm + pidx, Mx); store_partial(A.pl + pidx, Lc); }
#pragma unroll
      for (int c = 0; c < C; ++c) store_partial(A.pa + pidx * D + c0 + 64 * c + lane, Ac[c]);
    } else if (ns == 1) {      // the only partial of its rows: it is the result
#pragma unroll
      for (int c = 0; c < C; ++c) A.out[(qh0 + g) * D + c0 + 64 * c + lane] = __builtin_bit_cast(u16, (__bf16)(Lc > 0.f ? Ac[c] / Lc : 0.f));
    } else {
      if (lead) { ll_store(reinterpret_cast<u64*>(A.pm) + pidx, Mx, epoch); ll_store(reinterpret_cast<u64*>(A.pl) + pidx, Lc, epoch); }
#pragma unroll
      for (int c = 0; c < C; ++c) ll_store(reinterpret_cast<u64*>(A.pa) + pidx * D + c0 + 64 * c + lane, Ac[c], epoch);
    }
  };
  // two waves to a head while that is one pass, else one
  const auto merge_partials = [&](auto partials) {
    if (2 * G <= NW) { if (wave < 2 * G) merge_block(std::integral_constant<int, 1>{}, partials, wave >> 1, 64 * (wave & 1)); }
    else for (int g = wave; g < G; g += NW) merge_block(std::integral_constant<int, 2>{}, partials, g, 0);
  };
  if (RAWS > 1 && __builtin_amdgcn_readfirstlane(lds.two_raws)) merge_partials(std::integral_constant<int, NW + RAWS>{});
  else merge_partials(std::integral_constant<int, NW + 1>{});
  GAAC_STAMP(4);
  if (fused && A.nslot > 1 && ((rank >= 0 && ns > 1) || blockIdx.x == gridDim.x - 1)) {
    lds_barrier();      // every thread is done with the block-merge buffer, which becomes the mergers' scratch
    merge_heads<NW>(A, qh0, G, epoch, rec0, ns, rank, mergers, tid, *reinterpret_cast<MergeScratch<(NW > 8 ? 8 : NW)>*>(&M.acc[0][0][0]));
  }
  GAAC_STAMP(5);
}

// ---------------------------------------------------------------------------------------------------- split merge
__global__ void __launch_bounds__(512) k_attn_combine(const float* __restrict__ pm, const float* __restrict__ pl, const float* __restrict__ pa,
                                                      u16* __restrict__ out, int nslot) {
  __shared__ float fs[MAX_SLOTS];
  __shared__ float red[8];
  __shared__ float part[3][D];
  const int qh = blockIdx.x, tid = threadIdx.x, wv = tid >> 6;
  float m = -INFINITY;
  for (int s = tid; s < nslot; s += 512) m = fmaxf(m, pm[(long)qh * nslot + s]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((tid & 63) == 0) red[wv] = m;
  __syncthreads();
  float M = red[0];
#pragma unroll
  for (int w = 1; w < 8; ++w) M = fmaxf(M, red[w]);
  __syncthreads();
  float l = 0.f;
  for (int s = tid; s < nslot; s += 512) {
    const float v = pm[(long)qh * nslot + s];
    const float f = v == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(v - M);
    fs[s] = f; l += pl[(long)qh * nslot + s] * f;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
  if ((tid & 63) == 0) red[wv] = l;
  __syncthreads();
  float Lsum = 0.f;
#pragma unroll
  for (int w = 0; w < 8; ++w) Lsum += red[w];
  const int d = tid & 127, part_id = tid >> 7;      // four slot-interleaved partial sums per output element
  float acc = 0.f;
#pragma unroll 4
  for (int s = part_id; s < nslot; s += 4) acc += pa[((long)qh * nslot + s) * D + d] * fs[s];
  if (part_id) part[part_id - 1][d] = acc;
  __syncthreads();
  if (part_id == 0) {
    acc += part[0][d] + part[1][d] + part[2][d];
    const float o = Lsum > 0.f ? acc / Lsum : 0.f;
    out[(long)qh * D + d] = __builtin_bit_cast(u16, (__bf16)o);
  }
}

// ---------------------------------------------------------------------------------------------------- uncompressed baseline
// Decode attention over plain BF16 K/V [cache head][token][128] with the same structure as k_attn_split (same split / wave / MFMA
// mapping, online softmax, block merge and fused last-block merge) minus the decoder: the baseline the compressed path is compared
// with on the same GPU.  Args reuse AttnArgs: kt / vt = K / V, S_pad = token stride of a head, tcap = tokens per head.
struct RawTile { u32x4 k[4], v[4]; };
// K: lane (token a, quad q) holds channels 32 j + 8 q .. + 8 for product j.  V: lane (a, q) holds channels 8 a .. 8 a + 8 of tokens 4 q + r.
__device__ __forceinline__ void load_raw_tile(const u16* __restrict__ kh, const u16* __restrict__ vh, int tile, int S, int a, int q, RawTile& R) {
  const int kt = min(tile * T + a, S - 1);
#pragma unroll
  for (int j = 0; j < 4; ++j) R.k[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kh + (long)kt * D + 32 * j + 8 * q));
#pragma unroll
  for (int r = 0; r < 4; ++r) R.v[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vh + (long)min(tile * T + 4 * q + r, S - 1) * D + 8 * a));
}
template <bool PARTIAL>
__device__ __forceinline__ void consume_raw_tile(const RawTile& R, WaveState& st, int tile, int S, float scale_log2e, int q, const u32x4 (&qf)[4]) {
  f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j)
    sacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, R.k[j]), __builtin_bit_cast(bf16x8, qf[j]), sacc, 0, 0, 0);
  const int tok0 = tile * T + 4 * q;
  if (PARTIAL) {
#pragma unroll
    for (int r = 0; r < 4; ++r) sacc[r] = tok0 + r >= S ? -INFINITY : sacc[r];
  }
  const float tmax = quad_rows_max(fmaxf(fmaxf(sacc[0], sacc[1]), fmaxf(sacc[2], sacc[3])));
  if (__builtin_amdgcn_ballot_w64(tmax > st.m_run)) {
    const float mn = fmaxf(st.m_run, tmax), mu = mn == -INFINITY ? 0.f : mn * scale_log2e;
    const float alpha = __builtin_amdgcn_exp2f(st.m_run == -INFINITY ? -INFINITY : st.mu_run - mu);
    st.l_run *= alpha;
#pragma unroll
    for (int i = 0; i < 8; ++i) st.acc[i] *= alpha;
    st.m_run = mn; st.mu_run = mu;
  }
  float p[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[r], scale_log2e, -st.mu_run));
  st.l_run += (p[0] + p[1]) + (p[2] + p[3]);
  const u32x2 pw = {pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3])};
  const s16x4 pb = __builtin_bit_cast(s16x4, pw);
#pragma unroll
  for (int m = 0; m < 4; ++m) {      // word m of a row = channels 8 a + 2 m, + 1
    u32 w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = PARTIAL && tok0 + r >= S ? 0u : R.v[r][m];
    const u32x2 lo = {__builtin_amdgcn_perm(w[1], w[0], 0x05040100u), __builtin_amdgcn_perm(w[3], w[2], 0x05040100u)};
    const u32x2 hi = {__builtin_amdgcn_perm(w[1], w[0], 0x07060302u), __builtin_amdgcn_perm(w[3], w[2], 0x07060302u)};
    st.acc[2 * m] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, lo), pb, st.acc[2 * m], 0, 0, 0);
    st.acc[2 * m + 1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, hi), pb, st.acc[2 * m + 1], 0, 0, 0);
  }
}

// NW as in k_attn_split: eight-wave blocks (one per CU) for launches of up to 256 blocks, else four-wave blocks (two per CU)
template <int NW> struct Bf16Lds { u32x4 qw[GMAX][NG]; float m[NW][GMAX], l[NW][GMAX]; float acc[NW + 1][GMAX][D]; };      // acc: also the mergers' scratch
template <int NW>
__global__ void __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) k_bf16_attn_split(const AttnArgs A) {
  constexpr int NT = 64 * NW;
  __shared__ Bf16Lds<NW> L;
  const int bh = (int)blockIdx.x / A.nsplit, split = (int)blockIdx.x % A.nsplit, tid = threadIdx.x;      // a head's blocks are consecutive
  const int b = bh / A.n_kv, kvh = bh % A.n_kv, G = A.G;
  const long qh0 = (long)b * A.n_q + (long)kvh * G;
  const int S = A.sl ? min(max(A.sl[b], 0), A.tcap) : A.tcap;      // per-row lengths on the device (decode steps inside a graph) or one length
  const int ntiles = (S + T - 1) / T, chunk = (ntiles + A.nsplit - 1) / A.nsplit;
  const int tlo = min(split * chunk, ntiles), thi = min(tlo + chunk, ntiles);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, a = lane & 15, q = lane >> 4;
  const u16* kh = A.kt + (long)bh * A.S_pad * D; const u16* vh = A.vt + (long)bh * A.S_pad * D;
  // dynamic tile hand-out as in k_attn_split
  __shared__ int next_tile;
  const bool part_here = (S % T) != 0 && thi == ntiles && thi > tlo;
  const int thd = thi - (part_here ? 1 : 0), tcl = max(thd - 1, tlo);
  int tA = tlo + wave, tB = tA + NW;
  RawTile R0, R1;
  if (tA < thd) load_raw_tile(kh, vh, tA, S, a, q, R0);
  if (tid == 0) next_tile = tlo + 2 * NW;
  const u32 epoch = load_epoch(A);
  // Q as the B operand: lane (head a, quad q), product j covers channels 32 j + 8 q .. + 8 (rows >= G are zero)
  for (int i = tid; i < GMAX * NG; i += NT) {
    const int h = i >> 4, c = i & 15;
    L.qw[h][c] = h < G ? *reinterpret_cast<const u32x4*>(A.q + (qh0 + h) * D + 8 * c) : u32x4{0u, 0u, 0u, 0u};
  }
  __syncthreads();
  u32x4 qf[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) qf[j] = L.qw[a][4 * j + q];
  WaveState st;
#pragma unroll
  for (int i = 0; i < 8; ++i) st.acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  st.m_run = -INFINITY; st.mu_run = 0.f; st.l_run = 0.f;
  if (tA < thd) {
    while (true) {
      load_raw_tile(kh, vh, min(tB, tcl), S, a, q, R1);
      const int tC = uniform_tile(take_tile(&next_tile, thd, lane));
      consume_raw_tile<false>(R0, st, tA, S, A.scale_log2e, q, qf);
      if (tB >= thd) break;
      load_raw_tile(kh, vh, min(tC, tcl), S, a, q, R0);
      const int tD = uniform_tile(take_tile(&next_tile, thd, lane));
      consume_raw_tile<false>(R1, st, tB, S, A.scale_log2e, q, qf);
      if (tC >= thd) break;
      tA = tC; tB = tD;
    }
  }
  if (A.nslot > 1 && tid == 0) mark_arrival(A, epoch);
  if (part_here && wave == 0) {
    load_raw_tile(kh, vh, ntiles - 1, S, a, q, R0);
    consume_raw_tile<true>(R0, st, ntiles - 1, S, A.scale_log2e, q, qf);
  }
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
  const float l_run = quad_rows_sum(st.l_run);
  const float m_run = st.m_run == -INFINITY ? -INFINITY : st.mu_run;
  if (a < G) {
    if (q == 0) { L.m[wave][a] = m_run; L.l[wave][a] = l_run; }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) L.acc[wave][a][8 * (4 * q + r) + i] = st.acc[i][r];
  }
  lds_barrier();
  const int mergers = merge_ranks(G, A.nslot), rank = split - (A.nsplit - mergers);
  const int d = tid & 127;
  for (int g = tid >> 7; g < G; g += NT / 128) {
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, L.m[w][g]);
    float Lc = 0.f, Ac = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = L.m[w][g] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(L.m[w][g] - M);
      Lc += L.l[w][g] * f; Ac += L.acc[w][g][d] * f;
    }
    const long pidx = (qh0 + g) * A.nslot + split;
    if (A.nslot == 1) A.out[(qh0 + g) * D + d] = __builtin_bit_cast(u16, (__bf16)(Lc > 0.f ? Ac / Lc : 0.f));
    else {
      if (d == 0) { ll_store(reinterpret_cast<u64*>(A.pm) + pidx, M, epoch); ll_store(reinterpret_cast<u64*>(A.pl) + pidx, Lc, epoch); }
      ll_store(reinterpret_cast<u64*>(A.pa) + pidx * D + d, Ac, epoch);
    }
  }
  if (rank >= 0 && A.nslot > 1) {
    lds_barrier();
    merge_heads<NW>(A, qh0, G, epoch, qh0 * A.nslot, A.nslot, rank, mergers, tid, *reinterpret_cast<MergeScratch<NW>*>(&L.acc[0][0][0]));
  }
}

}  // namespace gaac

using namespace gaac;

// How many splits of n_kv blocks plan_block may count as resident, 0: no plan.  The plan costs a block about a microsecond at its start
// (its instructions come from memory on a first launch).  It cannot gain that
//   * where all blocks are resident and each row is one split, or a split of the longest possible row is no more than five tiles for
//     each of the block's eight waves, about 7 us;
//   * where one round is out of reach whatever the lengths, so that it only orders the rows, and there are many blocks of short rows: what
//     order can save is a split of the longest row at the end of the launch, the cost comes with every round.  One split per row, us
//     without and with the plan: 256 rows of up to 1000 tokens x 16 kv heads (4096 blocks, 67 tiles): 150 and 168, 256 of up to 2000 x
//     8 (2048, 129): 144 and 144, 128 of up to 4000 x 8 (1024, 254): 159 and 137.
// wide: the caller asked for more splits than the one round of eight-wave blocks that wide_splits left, so that an even share is what a long row loses by.
// Planned from two tiles a wave on (16 tiles a split) instead of five; us without and with the plan, with the store: 3 rows of 1400..6200 tokens x 8 kv heads
// 20.7 / 18.6, 5 of 400..2700 x 8 18.0 / 16.8, 8 of 190..1300 x 8 16.4 / 16.3, 2 of 3600..10500 x 4 17.6 / 16.7, 20 of 270..2900 x 2 18.6 / 17.4; alike rows pay the
// plan's start, 2 of 13000..14000 x 4 18.6 / 19.3, 8 of 1400..1500 x 8 17.3 / 18.0 (22.9 and 21.9 in four-wave blocks, planned).  From one tile a wave on nothing changes further.
constexpr long WIDE_PLAN = 16;
static int plan_units(int B, int n_kv, int nsplit, long max_tiles, bool wide = false) {
  const long blocks = (long)B * n_kv * nsplit;
  const int units = std::max((blocks > 256 ? 512 : 256) / n_kv, 1);
  if (B <= 1 || B > PLAN_ROWS || blocks >= SMALL_DIV) return 0;
  if (blocks <= 256) return nsplit > 1 && max_tiles > (wide ? WIDE_PLAN : 40l) * nsplit ? units : 0;
  if (nsplit > 1 && units >= B) return units;
  return 8 * max_tiles >= blocks * nsplit ? units : 0;
}

// A single row has nothing to share out: its splits are of one length, and where they are more than eight-wave blocks fit the chip, the second round, or half of one, comes
// on top.  Paged, one row of 65536 tokens, us, splits as of choose_nsplit / these / twice as many: 8 kv heads of 4 query heads 73 (256 splits) / 37.6 (32) / 37.9, 4 of
// 6 46.6 / 24.6 / 27.6, 2 of 8 27.6 / 19.4 / 27.6, 16 of 2 98 (128) / 65.8 / 65.1; of 16000 tokens 19.2 (62) / 17.2, 13.9 (62, as asked), 13.2 (as asked), 34.5 (62) / 23.5 / 22.8.
// That holds with CUs left over as well (wide_splits is for rows that are shared out, which gain from more blocks): as asked / these, of 2000, 8000 and 32000 tokens, 52 heads
// of 2 query heads (208 CUs) 17.6 / 16.3, 52 / 35, 126 / 110; 72 (216) 18.0 / 18.3, 63 / 43, 160 / 146; 96 (192) 27 / 22, 75 / 59, 205 / 203; 110 (220) 32 / 22, 80 / 60, 231 / 218.
// From 129 heads on that would be one split a head, and the blocks of long rows are better the smaller ones, two to a CU, in one round if that is
// nearly full or the row is short; as asked / one split / these, of 700, 2000, 8000 and 24000 tokens: 129 heads 19 / 17 / 17, 34 / 33 / 27, 89 / 104 / 74, 204 / 337 / 204; 160
// 19 / 17 / 17, 41 / 34 / 27, 102 / 110 / 81, 249 / 341 / 228; 200 19 / 17 / 17, 49 / 35 / 35, 119 / 107 / 106, 302 / 353 / 302; 256 20 / 18 / 18, 62 / 38 / 38, 144 / 123 / 122, 377 / 388 /
// 354; 320 29 / 25 / 25, 70 / 57 / 57, 175 / 199 / 175, 476 / 680 / 476; 512 37 / 28 / 28, 89 / 66 / 66, 259 / 238 / 238, 718 / 783 / 718.
static long single_row_splits(int n_kv, int nsplit, long max_tiles) {
  if (n_kv <= 128) return 256 / n_kv;
  const long n = 512 / n_kv;                                              // splits of four-wave blocks that fit the chip: 3, 2, 1, 0
  if (max_tiles <= 128) return n == 3 && nsplit >= 3 ? 3 : 1;             // (two splits of 129 heads are four-wave blocks too, but hardly more than CUs)
  const bool one_round = max_tiles <= 640 ? n >= 2 || (n == 1 && n_kv >= 384) : n >= 2 && n * n_kv >= 448;
  return one_round ? n : nsplit;
}
// Splits of a planned launch: no more than twice the resident blocks' worth.  A plan of one round leaves the other blocks without a part, and they start,
// look at the rows and are waited for behind the others; of several rounds, two do, as a row that needs more splits than the others gets them (SIZED_SPLIT).
// Paged, 8 kv heads, us, the caller's splits / these: 32 rows of 500..20000 tokens, 8 splits 168 / 166, 24 splits 181 / 165; 16 of 9000..11000 92 / 88, 20 of
// 39000..40000 405 / 385; 128 of 100..4000 x 4 heads, 4 splits 97 / 70; 64 of 2000, one of them 16000, 4 splits 120 / 111.
static int planned_splits(int B, int n_kv, int nsplit, int plan, long max_tiles, long least) {      // least: for splits that the paged kernel's tile table holds
  const long heads = (long)B * n_kv;
  if (B == 1) return (int)std::min<long>(nsplit, std::max(single_row_splits(n_kv, nsplit, max_tiles), least));
  return plan >= B ? (int)std::min<long>(nsplit, std::max((1024 + heads - 1) / heads, least)) : nsplit;
}

// Paged rows of few heads in all: splits for one round of eight-wave blocks, one per CU, where these fill it, instead of four-wave blocks, two per CU: half the
// starts, partials and records to wait for, and a wave has as many tiles.  us with the splits of choose_nsplit / these: 8 rows of 200..3000 tokens x 8 kv heads
// 18.1 / 16.4, 3 of 2900..3000 x 8 17.5 / 13.9, 9 of 39000..40000 x 4 93 / 88, 2 of 4000..60000 x 1 of 16 query heads 33.7 / 19.1, 39 of 1000 and one of 60000 x 1
// 32 / 20; 4 of 20000..60000 x 8 81.0 / 80.4.  The lines: with fewer CUs in use the gain is lost (52 heads on 208 CUs: 5000..40000 tokens 80.8 / 86.5, 96 on
// 192: 142 / 187), and four splits of long rows leave too little to even out: 64 heads, 4 rows of 20000..60000 147 / 158, of up to 10000 all 3 to 12 % faster.
static int wide_splits(int B, int n_kv, int nsplit, long max_tiles, long least) {
  const long heads = (long)B * n_kv, n = 256 / std::max(heads, 1l);
  const bool wide = heads <= 40 ? n * heads >= 240 : heads <= 64 && n * heads >= 248 && max_tiles <= 640;
  return B > 1 && wide && n >= least ? (int)std::min<long>(nsplit, n) : nsplit;
}

// Splits of a launch whose length the host knows: those of nsplit that get tiles, at least MIN_HOST_TILES each (the caller's count is an upper
// bound here, as it is in a planned launch; it sizes the workspace).  Empty splits and splits of a tile or two are blocks that only start, publish
// and are waited for.  us with splits of 2 or 3 / 3 / 4 / 6 tiles: 1000 tokens x 8 kv heads 9.3 / 8.4 / 8.4 / 9.1, 300 x 8 8.3 / 7.6 / 7.5 / 8.0,
// 2000 x 4 of 6 query heads 10.2 / 9.0 / 8.8 / 9.3, 1000 x 1 of 16 11.2 / 11.6 / 9.2 / 9.5, 500 x 2 x 2 of 8 8.2 / 8.0 / 7.9 / 8.5.
constexpr int MIN_HOST_TILES = 4;
static int host_splits(int tiles, int nsplit) {
  const int chunk = std::max((tiles + nsplit - 1) / nsplit, MIN_HOST_TILES);
  return std::max((tiles + chunk - 1) / chunk, 1);
}

#ifdef GAAC_PHASE_TIMING
static long long* g_dbg = nullptr;
extern "C" void gaac_set_phase_buffer(long long* p) { g_dbg = p; }
#endif
static int attn_split_impl(
    const uint8_t* smk, const uint8_t* ck, const int* fk, const int* tok, const uint8_t* ovk, const int* ohsk, const uint8_t* b3k, const uint8_t* b4k,
    const uint8_t* smv, const uint8_t* cv, const int* fv, const int* tov, const uint8_t* ovv, const int* ohsv, const uint8_t* b3v, const uint8_t* b4v,
    const void* q, const int* slot, int B, int n_q, int n_kv, const int* SL, int S_pad, float scale, int nsplit, int NB,
    const void* kt, const void* vt, const int* TL, int TCAP, void* pm, void* pl, void* pa, unsigned int* epoch, void* out, int S_all, void* stream) {
  GAAC_REQUIRE(n_kv > 0 && n_q > 0 && n_q % n_kv == 0 && n_q / n_kv >= 1 && n_q / n_kv <= GMAX, "GQA group size must be 1..%d (n_q=%d, n_kv=%d)", GMAX, n_q, n_kv);
  GAAC_REQUIRE(smk && ck && fk && tok && ovk && ohsk && b3k && b4k && smv && cv && fv && tov && ovv && ohsv && b3v && b4v, "gaac_attn: null store pointer");
  GAAC_REQUIRE(q && (SL || S_all >= 0) && pm && pl && pa, "gaac_attn: null pointer");
  GAAC_REQUIRE(S_all <= S_pad, "gaac_attn: S_all %d exceeds the token stride %d", S_all, S_pad);
  GAAC_REQUIRE(B > 0 && S_pad > 0 && S_pad % T == 0 && NB > 0, "gaac_attn: bad sizes B=%d S_pad=%d NB=%d", B, S_pad, NB);
  const bool has_tail = kt != nullptr;
  GAAC_REQUIRE(!has_tail || (vt && TL && TCAP >= 1 && TCAP <= T), "gaac_attn: tail needs kt, vt, TL and 1 <= TCAP <= %d", T);
  GAAC_REQUIRE(nsplit >= 1 && nsplit <= MAX_SLOTS, "gaac_attn: nsplit must be in 1..%d", MAX_SLOTS);
  GAAC_REQUIRE(S_pad > 0 && S_pad <= (1 << 24), "gaac_attn: at most %d tokens per cache head (32-bit byte offsets inside a head)", 1 << 24);
  if (epoch && S_all >= 0) nsplit = host_splits((S_all + T - 1) / T, nsplit);
  const int plan = epoch && S_all < 0 ? plan_units(B, n_kv, nsplit, S_pad / T) : 0;
  if (epoch && S_all < 0) nsplit = planned_splits(B, n_kv, nsplit, plan, S_pad / T, 1);
  const int nslot = nsplit;
  AttnArgs A;
  A.k = StoreView{smk, ck, fk, tok, ovk, ohsk, b3k, b4k};
  A.v = StoreView{smv, cv, fv, tov, ovv, ohsv, b3v, b4v};
  A.q = (const u16*)q; A.pm = (float*)pm; A.pl = (float*)pl; A.pa = (float*)pa; A.slot = slot; A.sl = SL; A.S_all = S_all < 0 ? -1 : S_all;
  A.S_pad = S_pad; A.scale_log2e = scale * 1.4426950408889634f; A.nsplit = nsplit; A.nslot = nslot;
  A.n_kv = n_kv; A.n_q = n_q; A.G = n_q / n_kv; A.NB = NB;
  A.kt = (const u16*)kt; A.vt = (const u16*)vt; A.tl = TL; A.tcap = TCAP;
  A.epochs = epoch; A.out = (u16*)out;
  A.B = B; A.plan = plan;
  GAAC_REQUIRE(!epoch || out, "gaac_attn: the fused merge needs an output buffer");
  A.pool = nullptr; A.raw = nullptr; A.mt = nullptr; A.bt = nullptr; A.bt_stride = 0; A.TS = 0;
  A.freeq = nullptr; A.n_free = 0; A.stack = nullptr; A.top = nullptr;
#ifdef GAAC_PHASE_TIMING
  A.dbg = g_dbg;
#endif
  // few blocks: one 8-wave block per CU (half as many partials); otherwise two 4-wave blocks per CU
  const bool wide = (long)B * n_kv * nslot <= 256;
  const dim3 grid(B * n_kv * nslot), block(wide ? 512 : 256);
#ifdef GAAC_WAVES12
  if (wide && S_all >= 0) hipLaunchKernelGGL((k_attn_split<false, 12, true>), grid, dim3(768), 0, (hipStream_t)stream, A);
#else
  if (wide && S_all >= 0) hipLaunchKernelGGL((k_attn_split<false, 8, true>), grid, block, 0, (hipStream_t)stream, A);
#endif
  else if (wide) hipLaunchKernelGGL((k_attn_split<false, 8, false>), grid, block, 0, (hipStream_t)stream, A);
  else if (S_all >= 0) hipLaunchKernelGGL((k_attn_split<false, 4, true>), grid, block, 0, (hipStream_t)stream, A);
  else hipLaunchKernelGGL((k_attn_split<false, 4, false>), grid, block, 0, (hipStream_t)stream, A);
  return launch_status("gaac_attn(split)");
}

extern "C" int gaac_attn_split(
    const uint8_t* smk, const uint8_t* ck, const int* fk, const int* tok, const uint8_t* ovk, const int* ohsk, const uint8_t* b3k, const uint8_t* b4k,
    const uint8_t* smv, const uint8_t* cv, const int* fv, const int* tov, const uint8_t* ovv, const int* ohsv, const uint8_t* b3v, const uint8_t* b4v,
    const void* q, const int* slot, int B, int n_q, int n_kv, const int* SL, int S_pad, float scale, int nsplit, int NB,
    const void* kt, const void* vt, const int* TL, int TCAP, float* pm, float* pl, float* pa, void* stream) {
  return attn_split_impl(smk, ck, fk, tok, ovk, ohsk, b3k, b4k, smv, cv, fv, tov, ovv, ohsv, b3v, b4v, q, slot, B, n_q, n_kv, SL, S_pad,
                         scale, nsplit, NB, kt, vt, TL, TCAP, pm, pl, pa, nullptr, nullptr, -1, stream);
}

extern "C" int gaac_attn_combine(const float* pm, const float* pl, const float* pa, void* out, int n_rows, int nslot, void* stream) {
  GAAC_REQUIRE(pm && pl && pa && out && n_rows > 0 && nslot >= 1 && nslot <= MAX_SLOTS, "gaac_attn_combine: bad arguments");
  hipLaunchKernelGGL(k_attn_combine, dim3(n_rows), dim3(512), 0, (hipStream_t)stream, pm, pl, pa, (u16*)out, nslot);
  return launch_status("gaac_attn(combine)");
}

extern "C" int gaac_attn_launch(
    const uint8_t* smk, const uint8_t* ck, const int* fk, const int* tok, const uint8_t* ovk, const int* ohsk, const uint8_t* b3k, const uint8_t* b4k,
    const uint8_t* smv, const uint8_t* cv, const int* fv, const int* tov, const uint8_t* ovv, const int* ohsv, const uint8_t* b3v, const uint8_t* b4v,
    const void* q, const int* slot, int B, int n_q, int n_kv, const int* SL, int S_pad, float scale, int nsplit, int NB,
    const void* kt, const void* vt, const int* TL, int TCAP,
    float* pm, float* pl, float* pa, void* out, void* stream) {
  GAAC_REQUIRE(out, "gaac_attn_launch: null output");
  int rc = attn_split_impl(smk, ck, fk, tok, ovk, ohsk, b3k, b4k, smv, cv, fv, tov, ovv, ohsv, b3v, b4v, q, slot, B, n_q, n_kv, SL, S_pad,
                           scale, nsplit, NB, kt, vt, TL, TCAP, pm, pl, pa, nullptr, nullptr, -1, stream);
  if (rc) return rc;
  return gaac_attn_combine(pm, pl, pa, out, B * n_q, nsplit, stream);
}

extern "C" int gaac_attn_fused(
    const uint8_t* smk, const uint8_t* ck, const int* fk, const int* tok, const uint8_t* ovk, const int* ohsk, const uint8_t* b3k, const uint8_t* b4k,
    const uint8_t* smv, const uint8_t* cv, const int* fv, const int* tov, const uint8_t* ovv, const int* ohsv, const uint8_t* b3v, const uint8_t* b4v,
    const void* q, const int* slot, int B, int n_q, int n_kv, const int* SL, int S_pad, float scale, int nsplit, int NB,
    const void* kt, const void* vt, const int* TL, int TCAP, int S_all,
    unsigned long long* pm, unsigned long long* pl, unsigned long long* pa, unsigned int* epoch, void* out, void* stream) {
  GAAC_REQUIRE(out && epoch, "gaac_attn_fused: null output or epoch buffer");
  return attn_split_impl(smk, ck, fk, tok, ovk, ohsk, b3k, b4k, smv, cv, fv, tov, ovv, ohsv, b3v, b4v, q, slot, B, n_q, n_kv, SL, S_pad,
                         scale, nsplit, NB, kt, vt, TL, TCAP, pm, pl, pa, epoch, out, S_all, stream);
}

// ---- the one entry point that allocates nothing ------------------------------------------------------------------------------------
// gaac_attn_fused with its workspace (partial records + epoch words) in a file-scope device array instead of caller memory, for callers
// that cannot allocate: code under HIP graph capture, tight serving loops.  Every GPU the library runs on holds its own copy of the
// array (4 MiB) from module load to process end; its address on a device comes from hipGetSymbolAddress, once per device
// (gaac_static_init, or the first call on that device outside stream capture).
constexpr size_t STATIC_SCRATCH_BYTES = 4u << 20;
constexpr long STATIC_MAX_RECORD_ROWS = 4000;                                               // B*n_q*nsplit (and so the grid's blocks) at most
constexpr size_t STATIC_EPOCH_BYTES = ((EPOCH_WORDS + STATIC_MAX_RECORD_ROWS) * sizeof(u32) + 255) / 256 * 256;      // epoch words + arrival marks
static_assert(STATIC_EPOCH_BYTES + STATIC_MAX_RECORD_ROWS * (D + 2) * sizeof(u64) <= STATIC_SCRATCH_BYTES, "the built-in workspace holds 4000 partial rows");
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];              // zero at module load: epoch 0, no records
constexpr int STATIC_MAX_DEVICES = 64;
static std::atomic<void*> g_scratch_ptr[STATIC_MAX_DEVICES];      // the array's address on each device (the name `scratch` is not one in host code)
static std::mutex g_scratch_mutex;

// The device a call runs on: the stream's own device when it has one, else the calling thread's current device.
static int static_device_of(hipStream_t stream, int* dev) {
  hipDevice_t d = -1;
  hipError_t e = stream ? hipStreamGetDevice(stream, &d) : hipGetDevice(&d);
  if (e != hipSuccess || d < 0 || d >= STATIC_MAX_DEVICES) return gaac::fail("gaac static workspace: no usable device (%s)", hipGetErrorString(e));
  *dev = (int)d;
  return 0;
}
// Resolves (once per device, under a lock) and returns the array's address on `dev`; dev must be the calling thread's current device.
static int static_scratch(int dev, bool may_resolve, unsigned char** base) {
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    if (!may_resolve)
      return gaac::fail("gaac_attn_fused_static: the built-in workspace of device %d has not been set up and the stream is capturing; "
                        "call gaac_static_init() once before the capture", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (!p) {
      int cur = -1;
      hipError_t e = hipGetDevice(&cur);
      if (e != hipSuccess || cur != dev) return gaac::fail("gaac static workspace: device %d is not the calling thread's current device (%d)", dev, cur);
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !p) return gaac::fail("gaac static workspace: hipGetSymbolAddress failed (%s)", hipGetErrorString(e));
      g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
  }
  *base = static_cast<unsigned char*>(p);
  return 0;
}

extern "C" int gaac_static_init(void) {
  int dev = -1;
  if (int rc = static_device_of(nullptr, &dev)) return rc;
  unsigned char* base = nullptr;
  return static_scratch(dev, true, &base);
}

__global__ void __launch_bounds__(256) k_fill_zero(u32x4* __restrict__ p, long n16) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n16) p[i] = u32x4{0u, 0u, 0u, 0u};
}
// Re-arms the built-in workspace of the stream's device after a failed launch: epoch words and records back to zero, by a kernel (not
// a memset node, so the call may be captured).
extern "C" int gaac_static_reset(void* stream) {
  int dev = -1;
  if (int rc = static_device_of((hipStream_t)stream, &dev)) return rc;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (stream && hipStreamIsCapturing((hipStream_t)stream, &cs) != hipSuccess) cs = hipStreamCaptureStatusNone;
  unsigned char* base = nullptr;
  if (int rc = static_scratch(dev, cs == hipStreamCaptureStatusNone, &base)) return rc;
  const long n16 = (long)(STATIC_SCRATCH_BYTES / 16);
  hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, reinterpret_cast<u32x4*>(base), n16);
  return launch_status("gaac_static_reset");
}
// Failure bits of the built-in workspace of the stream's device (see gaac_attn_fused), copied to *flags_out (device memory) on the stream.
extern "C" int gaac_static_flags(unsigned int* flags_out, void* stream) {
  GAAC_REQUIRE(flags_out, "gaac_static_flags: null output");
  int dev = -1;
  if (int rc = static_device_of((hipStream_t)stream, &dev)) return rc;
  unsigned char* base = nullptr;
  if (int rc = static_scratch(dev, true, &base)) return rc;
  hipError_t e = hipMemcpyAsync(flags_out, base + sizeof(unsigned int), sizeof(unsigned int), hipMemcpyDeviceToDevice, (hipStream_t)stream);
  if (e != hipSuccess) return gaac::fail("gaac_static_flags: %s", hipGetErrorString(e));
  return 0;
}

extern "C" int gaac_attn_fused_static(
    const uint8_t* smk, const uint8_t* ck, const int* fk, const int* tok, const uint8_t* ovk, const int* ohsk, const uint8_t* b3k, const uint8_t* b4k,
    const uint8_t* smv, const uint8_t* cv, const int* fv, const int* tov, const uint8_t* ovv, const int* ohsv, const uint8_t* b3v, const uint8_t* b4v,
    const void* q, const int* slot, int B, int n_q, int n_kv, const int* SL, int S_pad, float scale, int nsplit, int NB,
    const void* kt, const void* vt, const int* TL, int TCAP, int S_all, void* out, void* stream) {
  GAAC_REQUIRE(out, "gaac_attn_fused_static: null output");
  GAAC_REQUIRE(B > 0 && n_q > 0 && nsplit >= 1, "gaac_attn_fused_static: bad sizes B=%d n_q=%d nsplit=%d", B, n_q, nsplit);
  const long rec_rows = (long)B * n_q * nsplit;
  GAAC_REQUIRE(rec_rows <= STATIC_MAX_RECORD_ROWS,
               "gaac_attn_fused_static: B*n_q*nsplit = %ld exceeds the %ld partial rows the built-in workspace (%zu bytes) holds; use gaac_attn_fused with caller memory",
               rec_rows, STATIC_MAX_RECORD_ROWS, STATIC_SCRATCH_BYTES);
  int dev = -1;
  if (int rc = static_device_of((hipStream_t)stream, &dev)) return rc;
  unsigned char* base = g_scratch_ptr[dev].load(std::memory_order_acquire) ? static_cast<unsigned char*>(g_scratch_ptr[dev].load(std::memory_order_acquire)) : nullptr;
  if (!base) {      // first call on this device: resolve the address now, unless the stream is capturing (no runtime query inside a capture)
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (stream && hipStreamIsCapturing((hipStream_t)stream, &cs) != hipSuccess) cs = hipStreamCaptureStatusNone;
    if (int rc = static_scratch(dev, cs == hipStreamCaptureStatusNone, &base)) return rc;
  }
  unsigned int* epoch = reinterpret_cast<unsigned int*>(base);
  unsigned long long* pm = reinterpret_cast<unsigned long long*>(base + STATIC_EPOCH_BYTES);
  unsigned long long* pl = pm + rec_rows;
  unsigned long long* pa = pl + rec_rows;
  return attn_split_impl(smk, ck, fk, tok, ovk, ohsk, b3k, b4k, smv, cv, fv, tov, ovv, ohsv, b3v, b4v, q, slot, B, n_q, n_kv, SL, S_pad,
                         scale, nsplit, NB, kt, vt, TL, TCAP, pm, pl, pa, epoch, out, S_all, stream);
}

extern "C" int gaac_paged_attn(
    const uint8_t* pool, int TS, const void* raw, const int* mt, const int* bt, int bt_stride, const int* seq_lens, int max_seq_len,
    const void* q, int B, int n_q, int n_kv, float scale, int nsplit,
    const uint8_t* b3k, const uint8_t* b4k, const uint8_t* b3v, const uint8_t* b4v, int NB,
    unsigned long long* pm, unsigned long long* pl, unsigned long long* pa, unsigned int* epoch, void* out,
    const int* freeq, int n_free, int* stack, int* top, void* stream) {
  GAAC_REQUIRE(n_kv > 0 && n_q > 0 && n_q % n_kv == 0 && n_q / n_kv <= GMAX, "GQA group size must be 1..%d (n_q=%d, n_kv=%d)", GMAX, n_q, n_kv);
  GAAC_REQUIRE(!freeq || (n_free > 0 && stack && top), "gaac_paged_attn: a free queue needs its length, the stack and its top");
  GAAC_REQUIRE(pool && raw && mt && bt && seq_lens && q && b3k && b4k && b3v && b4v && pm && pl && pa && epoch && out, "gaac_paged_attn: null pointer");
  GAAC_REQUIRE(B > 0 && NB > 0 && TS >= SLOT_OV + 16 && TS % 16 == 0 && bt_stride > 0, "gaac_paged_attn: bad sizes B=%d NB=%d TS=%d (a slot is %d bytes plus at least 16 for escapes)", B, NB, TS, SLOT_OV);
  GAAC_REQUIRE(nsplit >= 1 && nsplit <= MAX_SLOTS, "gaac_paged_attn: nsplit must be in 1..%d", MAX_SLOTS);
  const long max_tiles = ((long)max_seq_len + T - 1) / T;
  GAAC_REQUIRE(max_seq_len >= 0 && max_tiles <= (long)bt_stride, "gaac_paged_attn: max_seq_len %d needs %ld blocks per row, the block table has %d", max_seq_len, max_tiles, bt_stride);
  const long least = (max_tiles + MAX_CHUNK - 1) / MAX_CHUNK;
  const int cut = wide_splits(B, n_kv, nsplit, max_tiles, least);
  const int plan = plan_units(B, n_kv, cut, max_tiles, cut < nsplit);
  nsplit = cut;
  nsplit = planned_splits(B, n_kv, nsplit, plan, max_tiles, least);
  AttnArgs A;
  A.k = StoreView{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, b3k, b4k};
  A.v = StoreView{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, b3v, b4v};
  A.q = (const u16*)q; A.pm = (float*)pm; A.pl = (float*)pl; A.pa = (float*)pa; A.slot = nullptr; A.sl = seq_lens; A.S_all = -1;
  A.S_pad = 0; A.scale_log2e = scale * 1.4426950408889634f; A.nsplit = nsplit; A.nslot = nsplit;
  A.n_kv = n_kv; A.n_q = n_q; A.G = n_q / n_kv; A.NB = NB;
  A.kt = nullptr; A.vt = nullptr; A.tl = nullptr; A.tcap = 0;
  A.epochs = epoch; A.out = (u16*)out;
  A.B = B; A.plan = plan;
  A.pool = pool; A.raw = (const u16*)raw; A.mt = mt; A.bt = bt; A.bt_stride = bt_stride; A.TS = TS;
  A.freeq = freeq; A.n_free = freeq ? n_free : 0; A.stack = stack; A.top = top;
#ifdef GAAC_PHASE_TIMING
  A.dbg = g_dbg;
#endif
  if ((long)B * n_kv * nsplit <= 256) hipLaunchKernelGGL((k_attn_split<true, 8, false>), dim3(B * n_kv * nsplit), dim3(512), 0, (hipStream_t)stream, A);
  else hipLaunchKernelGGL((k_attn_split<true, 4, false>), dim3(B * n_kv * nsplit), dim3(256), 0, (hipStream_t)stream, A);
  return launch_status("gaac_paged_attn");
}

extern "C" int gaac_bf16_attn(const void* k, const void* v, int S, const int* seq_lens, long head_stride_tokens, const void* q, int B, int n_q,
                              int n_kv, float scale, int nsplit, unsigned long long* pm, unsigned long long* pl, unsigned long long* pa,
                              unsigned int* epoch, void* out, void* stream) {
  GAAC_REQUIRE(n_kv > 0 && n_q > 0 && n_q % n_kv == 0 && n_q / n_kv <= GMAX, "GQA group size must be 1..%d (n_q=%d, n_kv=%d)", GMAX, n_q, n_kv);
  GAAC_REQUIRE(k && v && q && pm && pl && pa && epoch && out, "gaac_bf16_attn: null pointer");
  GAAC_REQUIRE(B > 0 && S > 0 && head_stride_tokens >= S && nsplit >= 1 && nsplit <= MAX_SLOTS, "gaac_bf16_attn: bad sizes");
  AttnArgs A = {};
  A.q = (const u16*)q; A.pm = (float*)pm; A.pl = (float*)pl; A.pa = (float*)pa; A.S_all = -1;
  A.S_pad = (int)head_stride_tokens; A.scale_log2e = scale * 1.4426950408889634f; A.nsplit = nsplit; A.nslot = nsplit;
  A.n_kv = n_kv; A.n_q = n_q; A.G = n_q / n_kv; A.NB = 1;
  A.kt = (const u16*)k; A.vt = (const u16*)v; A.tcap = S; A.sl = seq_lens;
  A.epochs = epoch; A.out = (u16*)out;
  if ((long)B * n_kv * nsplit <= 256) hipLaunchKernelGGL(k_bf16_attn_split<8>, dim3(B * n_kv * nsplit), dim3(512), 0, (hipStream_t)stream, A);
  else hipLaunchKernelGGL(k_bf16_attn_split<4>, dim3(B * n_kv * nsplit), dim3(256), 0, (hipStream_t)stream, A);
  return launch_status("gaac_bf16_attn");
}
