// Device-side helpers shared by the attention forward and backward kernels.
//
// Register layouts used throughout (wave64, gfx950), verified on hardware:
//   v_mfma_f32_32x32x16 A (32 x 16): lane l holds row l%32, k = 8*(l/32) .. +7
//                       B (16 x 32): lane l holds col l%32, k = 8*(l/32) .. +7
//                       C (32 x 32): lane l holds col l%32, reg i is row
//                                    8*(i/4) + 4*(l/32) + i%4
//   ds_read_b64_tr_b16: within each group of 16 lanes, lane i supplies the
//                       address of 4 consecutive 16-bit elements; it receives
//                       element i%4 of lanes (i/4), 4+(i/4), 8+(i/4), 12+(i/4),
//                       i.e. column i of the 4 x 16 block whose row r is the
//                       concatenation of lanes 4r .. 4r+3.
#pragma once

#include "rswa_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace rswa {

constexpr float kLog2e = 1.4426950408889634f;

// Division of 0 <= n < 2^31 by a launch constant as a multiplication and a shift (a division by a value
// the compiler does not know is some 30 dependent instructions, five of them ahead of a block's first
// load).  The method is Granlund and Montgomery's ("Division by Invariant Integers using Multiplication",
// 1994): multiplier 2^32 + mul with mul = floor(2^32 (2^shift - d) / d) + 1, shift = ceil(log2 d).
// (`d` is read of the walk's period only; in the others it keeps the kernel arguments behind where they load best:
// without it a forward of 2 x 333 rows, 8 / 2 heads, fp16, took 9.44 us instead of 9.33.)
struct FastDiv {
  uint32_t d, mul, shift;
};
inline FastDiv fast_div(uint32_t d) {  // d >= 1
  uint32_t s = 0;
  while ((1ull << s) < d) s++;
  return {d, (uint32_t)(((1ull << 32) * ((1ull << s) - d)) / d + 1), s};
}
__host__ __device__ __forceinline__ int quotient(int n, const FastDiv& f) {
  return (int)(((uint32_t)((uint64_t)(uint32_t)n * f.mul >> 32) + (uint32_t)n) >> f.shift);
}

// Kernel-side view of rswa_attn_params (strides in elements).
struct AttnArgs {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;
  const void* dout;
  void* dq;
  void* dk;
  void* dv;
  float* delta;   // fp32 [heads_q, rows_q] packed: -sum_d dO * O         (workspace)
  float* lse2;    // fp32 [heads_q, rows_q] packed: -lse * log2(e); empty rows -inf (workspace)
  int32_t n_count;    // arrival counters in the workspace (sink kernel)
  // backward of a pack (workspace; null: no table): number of dK/dV key tiles before sequence b, for
  // b = 0 .. batch, then whether the blocks take the snake order; written ahead of the dK/dV launch
  // by a kernel of the same call; a tile has 2^ktile_log2 keys
  int32_t* ktile;
  int32_t ktile_log2;
  int32_t snake;    // dK/dV: see the kernel (dense; of a pack the device decides)
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t q_st[3], k_st[3], v_st[3], o_st[3], do_st[3], dq_st[3], dk_st[3], dv_st[3], lse_st[3];
  int64_t rows_q;  // batch * seqlen_q (dense) or total_q (packed)
  int64_t rows_k;  // batch * seqlen_k (dense) or total_k (packed)
  int32_t batch, heads_q, heads_kv, group;  // group = heads_q / heads_kv
  int32_t seqlen_q, seqlen_k;
  int32_t wl, wr, n_sink;  // wl/wr < 0: unbounded
  int32_t shift_explicit, shift_val;
  int32_t dq_accumulate;  // backward: add to dq instead of overwriting it
  int32_t out_accumulate;  // forward: merge the block into what out / lse hold
  // fp32 / fp64 accumulators of the ring loops in place of 16-bit / fp32 results (RSWA_WIDE_*):
  // forward out fp32 + lse fp64; backward dq fp32; backward dk, dv fp32 (+ add to them)
  int32_t wide_out, wide_dq, wide_dkv, dkv_accumulate;
  int32_t n_tile;          // tiles per sequence (dense) / total tile slots (packed)
  int32_t n_work;          // logical blocks
  int32_t xcd_log2, n_group, tile_heads;  // see tile_of_block; kv heads of all batch entries (a pack: kv heads)
  FastDiv by_tile, by_heads, by_units;  // n_tile, heads_kv, blocks per (kv head, tile)
  // Blocks are dispatched in logical order; these flags reverse the order of the query
  // tiles (forward, dQ) or key tiles (dK/dV) so that the tiles with the most visible
  // pairs start first and the short ones fill the tail of the launch.
  int32_t rev_q, rev_k;
  FastDiv by_walk;  // see KeyWalk
  // backward with sink keys and a bounded window: workspace of the sink kernel -- fp32 sums
  // [sequence x kv head][chunk of rows][sink][dK, dV][D] and one arrival counter per
  // (sequence, kv head); null when that kernel does not run
  float* sink_part;
  int32_t* sink_count;
  int32_t sink_chunks;  // row chunks per (sequence, kv head)
  // keys in two row ranges: key rows [0, seg) of k / v / dk / dv, the rest in k2 / v2 / dk2 / dv2
  // (same strides); seg = INT32_MAX when all keys lie in k / v
  const void* k2;
  const void* v2;
  void* dk2;
  void* dv2;
  int32_t seg;
  int32_t avg_keys;  // keys a query row sees on average (host estimate; block shapes hang on it)
  int32_t far;  // a sequence of some streamed tensor spans 2 GiB or more: FAR kernels
  // dS hand-off (backward): the dK/dV kernel stores its packed 16-bit dS tiles and the dQ
  // kernel of that route only multiplies them with K.  Unit = 32 query rows x 64 keys (one
  // wave's step), 4 KiB, at ds + (((q head * ds_slots + row-tile slot) * ds_nkb + key block %
  // ds_nkb) * 4 + 64-key group) * 4096; a row tile sees at most ds_nkb consecutive 256-key
  // blocks.  Null: the dQ kernel recomputes S and dP.
  char* ds;
  int32_t ds_nkb;
  int32_t ds_slots;  // 32-row tile slots per q head (dense: batch * tiles; packed: rows / 32 + batch)
  float scale, scale_log2;
  // ---- for the host's choices only; behind the rest, so that the kernels' argument loads stay put
  int32_t max_keys;   // keys a query row sees at most (of the rows avg_keys samples)
  int32_t dkdv_form;  // RSWA_DKDV_*: the caller's choice of the dK/dV kernel's blocks
  int32_t dq_last;    // dq lies over an input: the dQ kernel must not run before dK/dV
};

struct SeqInfo {
  int64_t q_row0, k_row0;  // first row of the sequence in the (batch-strided or packed) tensor
  int64_t q_base, k_base;  // element offset of the batch (dense) — 0 in packed mode
  int32_t len_q, len_k;
  int32_t batch_idx;
};

// Which tile (of all: kv head after kv head, batch entry after batch entry, n_tile each) and which of its
// `units` blocks is this block's?  Hardware deals block ids to the 8 XCDs in turn, and blocks that share K / V
// should share an L2.  xcd_log2 = 0: every XCD takes an eighth of all blocks in a row.  Else the XCDs form groups of
// 1 << xcd_log2, each with n_group tiles that its XCDs take in turn (see deal_blocks).  False: a block beyond the last.
__device__ __forceinline__ bool tile_of_block(const AttnArgs& a, int units, int& tile, int& unit) {
  const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
  if (a.xcd_log2 == 0) {
    const int id = x * ((int)gridDim.x >> 3) + j;
    tile = quotient(id, a.by_units);
    unit = id - tile * units;
    return id < a.n_work;
  }
  const int k = quotient(j, a.by_units);
  unit = j - k * units;
  const int at = (k << a.xcd_log2) + (x & ((1 << a.xcd_log2) - 1));
  tile = (x >> a.xcd_log2) * a.n_group + at;
  return at < a.n_group;
}

// XCDs (as a power of two) that share kv heads where each takes an eighth of them all: 0 if each has whole ones.
inline int xcds_per_head_log2(const AttnArgs& a) {
  const int heads = a.heads_kv * (a.cu_q ? 1 : a.batch);
  return 3 - std::min(3, (int)__builtin_ctz((unsigned)heads));
}
// Tile dealing for a.n_tile tiles per kv head (and batch entry) of `units` blocks each: sets what the kernels read
// and returns the blocks to launch.  `spread`: XCDs that share kv heads take their tiles in turn.
inline int64_t deal_blocks(AttnArgs& a, int units, bool spread) {
  const int64_t heads = (int64_t)a.heads_kv * (a.cu_q ? 1 : a.batch);
  a.xcd_log2 = spread ? xcds_per_head_log2(a) : 0;
  a.n_work = (int)(heads * a.n_tile * units);
  a.tile_heads = (int)heads;
  a.n_group = (int)((heads << a.xcd_log2 >> 3) * a.n_tile);  // (whole heads; xcd_log2 = 0: read where heads % 8 == 0)
  a.by_tile = fast_div((uint32_t)a.n_tile);
  a.by_heads = fast_div((uint32_t)a.heads_kv);
  a.by_units = fast_div((uint32_t)units);
  return a.xcd_log2 ? ceil_div(a.n_group, 1 << a.xcd_log2) * 8 * units : ceil_div(a.n_work, 8) * 8;
}
constexpr int kComputeUnits = 256;  // MI355X

// Should forward and dQ blocks be spread?  Tiles in a row share their windows' K and V, so an XCD with every second
// tile reads almost twice the bytes (12 = 12 heads, even work: 3 to 6 % slower); but where the rows of some parts of a
// sequence see fewer keys, parts make unequal eighths (us, eighths / spread: rank step of 7298 rows, 28 / 4 heads,
// window 5372, forward 429 / 348, dQ 651 / 524; 3958 rows, 28 / 4 heads, a sink, window 2397, 126 / 109 and 178 / 139;
// 2 x 18605 rows, 8 / 2 heads, head_dim 64, window 3149, 277 / 253 and 329 / 300).  So: where the fullest eighth has
// 5 % more than the average, of a dense call (of a pack the host knows too little, and both orders lost and won).  A
// row counts as its keys and 200 for starts and ends.  (123 drawn calls with such heads: forward 1.1 % and dQ 1.3 %
// faster than eighths on average, 23 % at most; nothing slower beyond the 7 % by which single calls scatter.)
inline bool spread_rows(const AttnArgs& a) {
  const int log2 = xcds_per_head_log2(a);
  const int heads = (a.heads_kv * a.batch) << log2 >> 3;  // that 1 << log2 XCDs share
  if (a.cu_q || log2 == 0 || heads > 8) return false;
  constexpr int S = 32;  // samples per head
  const int64_t sh = a.shift_explicit ? a.shift_val : (int64_t)a.seqlen_k - a.seqlen_q;
  int64_t before[S + 1] = {0};  // keys of a head's first samples
  for (int i = 0; i < S; i++) {
    const int64_t row = (int64_t)(2 * i + 1) * a.seqlen_q / (2 * S);
    const int64_t hi = a.wr >= 0 ? std::min<int64_t>(a.seqlen_k - 1, row + sh + a.wr) : a.seqlen_k - 1;
    const int64_t lo = a.wl >= 0 ? std::max<int64_t>(0, row + sh - a.wl) : 0;
    before[i + 1] = before[i] + std::max<int64_t>(0, hi - lo + 1) + 200;
  }
  // (a part is whole samples; every one of a loop over all heads' samples took up to 1.2 us of host time, 0.1 so)
  auto until = [&](int samples) { return samples / S * before[S] + before[samples % S]; };
  int64_t most = 0;
  for (int p = 0; p < 1 << log2; p++)
    most = std::max(most, until((p + 1) * heads * S >> log2) - until(p * heads * S >> log2));
  return (double)most * (1 << log2) > 1.05 * (double)until(heads * S);
}

// And dK/dV blocks?  Lengths vary more (keys at a sequence's end are seen by few rows), and with tiles in a row one
// XCD's last blocks are those of a sequence's end, short or long, and its share of a pack's sequences is what comes (us,
// dK/dV, eighths / spread: 28 / 4 heads, head_dim 64, 3914 rows against 5194 keys, window 1296, 122 / 90; rank step of
// 4667 rows, 12 = 12 heads, window 5365, 107 / 96; packs of 23745 tokens, 28 / 4 heads, window 2203, 679 / 630, and of
// 16544, 4 = 4 heads, window 1132, 99 / 92).  Not where windows are short against the sequences (even work) and the
// launch has a second round to even out what the first leaves (25429 rows, 16 / 4 heads, window 593, 400 blocks, 183 /
// 189; packs of long sequences, 8 / 2 heads, windows 90 and 205, 36 / 41 and 119 / 128; but 4134 rows, 28 / 4 heads,
// window 173, 260 blocks, 64 / 53, and 20516 rows, window 568, 324 blocks, 438 / 405).  480 drawn calls with such heads:
// the rule is 2.0 % faster than eighths on average (ranks' chunks 7 %, packs that a rank shares 3 %, the others 0.3 to 1.1 %;
// as many kv heads as q heads, 206 calls, 2.1 %), 100 calls by more than 3 % and 38 % at most; 42 are slower by more than
// 3 %, mostly packs, the worst of 64 and 70 short sequences (8104 tokens, 4 = 4 heads, 26.9 / 33.1; 5423, 16 / 4,
// head_dim 64, 21.5 / 27.0), where it depends on lengths that the host does not know.  Spreading always: 1.2 % faster on
// 240 of them where the rule is 1.6 %; packs by their number of sequences: 1.7 % on 240 others, the rule 2.4 %.
inline bool spread_keys(const AttnArgs& a) {
  const int64_t heads = (int64_t)a.heads_kv * (a.cu_q ? 1 : a.batch);
  const int64_t len = a.cu_q ? a.rows_k / a.batch : a.seqlen_k;
  const bool even = a.wl >= 0 && a.wr >= 0 && ((int64_t)a.wl + a.wr + 1) * 8 < len;
  return !even || heads * a.n_tile <= kComputeUnits * 7 / 5;
}

// Mask bounds of one query row i (local index): visible keys are
//   j <= hi  and  (j >= lo or j < n_sink);   hi already clipped to len_k - 1.
struct RowBounds {
  int lo, hi;
};

__host__ __device__ __forceinline__ RowBounds row_bounds(const AttnArgs& a, int i, int len_q, int len_k) {
  RowBounds r;
  const int shift = a.shift_explicit ? a.shift_val : len_k - len_q;
  r.hi = (a.wr >= 0) ? min(len_k - 1, i + shift + a.wr) : len_k - 1;
  r.lo = (a.wl >= 0) ? max(0, i + shift - a.wl) : 0;
  if (i >= len_q) r.hi = -1;  // rows past the end see nothing
  return r;
}

// The tiles of BN keys that a block of rows i0 .. i_last visits: those of the sink keys that lie before its rows'
// windows, from tile 0 on, then n_band from tile t_lo on.
struct KeyTiles {
  int n_sink, t_lo, n_band;
};
template <int BN>
__host__ __device__ __forceinline__ KeyTiles key_tiles(const AttnArgs& a, int i0, int i_last, int len_q, int len_k) {
  const int lo = row_bounds(a, i0, len_q, len_k).lo, hi = row_bounds(a, i_last, len_q, len_k).hi;
  const bool band = hi >= lo;
  KeyTiles t;
  t.t_lo = band ? lo / BN : (1 << 29);
  t.n_band = band ? hi / BN - t.t_lo + 1 : 0;
  const int sink_keys = max(0, min(min(a.n_sink, hi + 1), lo));
  t.n_sink = min((sink_keys + BN - 1) / BN, t.t_lo);
  return t;
}
// Their order: the sinks' tiles, then the band from its first tile on whose number is a multiple of a period, around its
// end.  Blocks that start together are then on few tiles at a time instead of one tile each: with as many kv heads as
// q heads the 64 blocks that an XCD runs at once cover 8192 rows, whose K and V are as large as its L2, and every
// block of a window found its tiles gone again.  2 x 8192 rows, 32 = 32 heads, head_dim 128, window 1000, walks from the
// first tile / from here: fetched beyond L2 in the forward 1.89 / 0.43 GB, in dQ 1.98 / 0.72 GB; a training call
// 1299 / 1243 us.
// No block has two multiples of the period (walk_period), so a row sees its tiles in an order that its window alone
// decides, whichever rows its block holds besides: from the multiple among them on, if there is one, else from the
// first (tiles that none of its keys lie in change nothing).  And hardly more tiles than a block has, so that few
// blocks have none: with the next power of two instead (no division ahead of a block's first load) the same call
// was 1.6 % slower, a forward of 2 x 11372 rows, 32 heads, window 142, 2 %.
//
// A cursor; advanced beyond the last tile it is on one of them still.  (A comparison and
// three selects a tile; computing a tile from its place in the walk, three times per tile in the forward, cost
// the launches that gain nothing from the order 1 % (24 drawn calls with equal heads: forward 0.4 % slower than
// with walks from the first tile that way, 1.8 % faster with the cursor; dQ 0.1 and 2.2 % faster).)
struct KeyWalk {
  int tile;        // where the cursor is
  int stop, jump;  // reaching tile `stop` it goes to tile `jump` ...
  int end, back;   // ... after which these take their place
  __host__ __device__ __forceinline__ KeyWalk(const AttnArgs& a, const KeyTiles& t) {
    const int at = quotient(t.t_lo + (int)a.by_walk.d - 1, a.by_walk) * (int)a.by_walk.d - t.t_lo;
    const int first = t.n_band > 0 ? t.t_lo + (at < t.n_band ? at : 0) : 0;
    end = t.n_band > 0 ? t.t_lo + t.n_band : t.n_sink;
    back = t.n_band > 0 ? t.t_lo : 0;
    tile = t.n_sink > 0 ? 0 : first;
    stop = t.n_sink > 0 ? t.n_sink : end;
    jump = t.n_sink > 0 ? first : back;
  }
  // BRANCH: by a branch that is taken once or twice a walk instead of selects, five instructions a tile (the dQ
  // kernel at head_dim 128, whose waves start a tile together and wait for it; the forward gains nothing)
  template <bool BRANCH>
  __host__ __device__ __forceinline__ void next() {
    tile++;
    if constexpr (BRANCH) {
      if (__builtin_expect(tile == stop, 0)) {
        asm volatile("");
        tile = jump;
        stop = end;
        jump = back;
      }
    } else {
      const bool at = tile == stop;
      tile = at ? jump : tile;
      stop = at ? end : stop;
      jump = at ? back : jump;
    }
  }
};
// The period for blocks of up to `block_rows` rows: the tiles of the largest band; and of the sinks, so that a band that
// begins among their tiles has no multiple behind them.
inline FastDiv walk_period(const AttnArgs& a, int block_rows, int tile_keys) {
  if (a.wl < 0 || a.wr < 0) return fast_div(1);  // (from the first tile)
  const int64_t band = ((int64_t)a.wl + a.wr + block_rows + tile_keys - 2) / tile_keys + 1;
  return fast_div((uint32_t)(band + ceil_div(a.n_sink, tile_keys)));
}

// Packed mode: which sequence, and which of its tiles of `tile` = 2^tile_log2 rows, does
// tile slot `t` along the q or k axis stand for?  Sequence b owns the slots from
// cu[b] / tile + b on -- strictly increasing in b, so a search over cu finds b, where a running
// count of tiles would have to walk every sequence before it.  The search goes 64 ways at a time (each
// lane tests one entry, the ballot counts those at or below t): one load deep up to 64 sequences, two up
// to 4096, where halving took a dependent load per factor of two, 7 of them ahead of a block's first
// load in a pack of 70 sequences.  Every lane takes part; the results are wave-uniform.
// ceil(len_b / tile) of its slots are its tiles; at most one more, before
// the next sequence's first, stays unused (false is returned for it), which is why a packed
// grid has ceil(rows / tile) + batch slots.
__device__ __forceinline__ bool locate_packed(const AttnArgs& a, int t, int tile_log2, bool along_k,
                                              SeqInfo& s, int& tile_in_seq) {
  const int32_t* cu = along_k ? a.cu_k : a.cu_q;
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  int lo = 0, n = a.batch;  // the sequence is one of lo .. lo + n - 1
  for (;;) {
    const int step = (n + 63) >> 6;
    const int i = min(lo + lane * step, lo + n - 1);
    const int slot = (cu[i] >> tile_log2) + i;
    const int at = max(__popcll(__builtin_amdgcn_ballot_w64(lane * step < n && slot <= t)) - 1, 0);
    lo += at * step;
    if (step == 1) break;
    n = min(step, n - at * step);
  }
  const int b = lo;
  const int first = cu[b];
  tile_in_seq = t - ((first >> tile_log2) + b);
  if ((tile_in_seq << tile_log2) >= cu[b + 1] - first) return false;
  s.batch_idx = b;
  s.q_row0 = a.cu_q[b];
  s.k_row0 = a.cu_k[b];
  s.len_q = a.cu_q[b + 1] - a.cu_q[b];
  s.len_k = a.cu_k[b + 1] - a.cu_k[b];
  s.q_base = 0;
  s.k_base = 0;
  return true;
}

// The same along k from the exact table a.ktile: tile number t (of a.ktile[batch]) is tile
// tile_in_seq of sequence s.  The search goes 64 ways at a time: each lane tests one entry, the
// ballot counts those at or below t.  Every lane takes part; the results are wave-uniform.
__device__ __forceinline__ void locate_tile(const AttnArgs& a, int t, SeqInfo& s, int& tile_in_seq) {
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  int lo = 0, n = a.batch;  // the sequence is one of lo .. lo + n - 1, and ktile[lo] <= t
  int c;
  for (;;) {
    const int step = (n + 63) >> 6;
    const int i = lo + lane * step;
    c = a.ktile[min(i, lo + n - 1)];
    const int at = __popcll(__builtin_amdgcn_ballot_w64(lane * step < n && c <= t)) - 1;
    lo += at * step;
    if (step == 1) {
      tile_in_seq = t - __builtin_amdgcn_readlane(c, at);
      break;
    }
    n = min(step, n - at * step);
  }
  s.batch_idx = lo;
  s.q_row0 = a.cu_q[lo];
  s.k_row0 = a.cu_k[lo];
  s.len_q = a.cu_q[lo + 1] - a.cu_q[lo];
  s.len_k = a.cu_k[lo + 1] - a.cu_k[lo];
  s.q_base = 0;
  s.k_base = 0;
}

template <typename T>
struct Mma;

template <>
struct Mma<__bf16> {
  using V8 = bf16x8;
  using V4 = bf16x4;
  static __device__ __forceinline__ f32x16 mfma32(V8 a, V8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(V8 a, V8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  // The same instruction as inline assembly with the accumulator kept in vector registers
  // (for accumulators the vector ALU reads next; the builtin's accumulators live in
  // accumulation registers), and a zero-initialising form (early clobber: the destination
  // of a 32x32 MFMA must not overlap its A / B operands).  The compiler sees opaque
  // statements and inserts no wait states after them: the caller keeps at least two later
  // MFMAs (or 32 idle cycles) between one of these and any other instruction that reads
  // its result, copies added by the register allocator included -- accumulators that live
  // across control flow are therefore better served by the builtin.  Volatile: they keep
  // their order among themselves and the empty volatile statements that pin vector work.
  // RSWA_MFMA_BUILTIN_ONLY builds the same three through the builtin instead: the compiler then
  // pads every hazard itself (and is free to place the accumulators badly).  The build makes a
  // second library that way, and a GPU test holds the two to the same output bits -- a
  // scheduler change in a later compiler that broke the distance kept by hand would show there.
#ifndef RSWA_MFMA_BUILTIN_ONLY
  static __device__ __forceinline__ void mfma32_vec(V8 a, V8 b, f32x16& c) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mfma32_vec0(V8 a, V8 b, f32x16& c) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
  }
  // first MFMA of a chain that starts from `init` instead of zero
  static __device__ __forceinline__ void mfma32_vec_init(V8 a, V8 b, const f32x16& init, f32x16& c) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(c) : "v"(a), "v"(b), "v"(init));
  }
#else
  static __device__ __forceinline__ void mfma32_vec(V8 a, V8 b, f32x16& c) { c = mfma32(a, b, c); }
  static __device__ __forceinline__ void mfma32_vec0(V8 a, V8 b, f32x16& c) {
    c = mfma32(a, b, f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0});
  }
  static __device__ __forceinline__ void mfma32_vec_init(V8 a, V8 b, const f32x16& init, f32x16& c) {
    c = mfma32(a, b, init);
  }
#endif
  static __device__ __forceinline__ V8 pack(const float* x) {
    f32x8 f = {x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]};
    return __builtin_convertvector(f, V8);
  }
  static __device__ __forceinline__ V4 pack4(float a, float b, float c, float d) {
    f32x4 f = {a, b, c, d};
    return __builtin_convertvector(f, V4);
  }
};

template <>
struct Mma<_Float16> {
  using V8 = f16x8;
  using V4 = f16x4;
  static __device__ __forceinline__ f32x16 mfma32(V8 a, V8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(V8 a, V8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
#ifndef RSWA_MFMA_BUILTIN_ONLY
  static __device__ __forceinline__ void mfma32_vec(V8 a, V8 b, f32x16& c) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ void mfma32_vec0(V8 a, V8 b, f32x16& c) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
  }
  // first MFMA of a chain that starts from `init` instead of zero
  static __device__ __forceinline__ void mfma32_vec_init(V8 a, V8 b, const f32x16& init, f32x16& c) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %3" : "=&v"(c) : "v"(a), "v"(b), "v"(init));
  }
#else
  static __device__ __forceinline__ void mfma32_vec(V8 a, V8 b, f32x16& c) { c = mfma32(a, b, c); }
  static __device__ __forceinline__ void mfma32_vec0(V8 a, V8 b, f32x16& c) {
    c = mfma32(a, b, f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0});
  }
  static __device__ __forceinline__ void mfma32_vec_init(V8 a, V8 b, const f32x16& init, f32x16& c) {
    c = mfma32(a, b, init);
  }
#endif
  static __device__ __forceinline__ V8 pack(const float* x) {
    f32x8 f = {x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]};
    return __builtin_convertvector(f, V8);
  }
  static __device__ __forceinline__ V4 pack4(float a, float b, float c, float d) {
    f32x4 f = {a, b, c, d};
    return __builtin_convertvector(f, V4);
  }
};

typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// XOR swizzle of 16-byte chunks inside an LDS tile whose rows hold CH chunks (8 or 16):
// chunk c of row r is stored at chunk position c ^ swz_f<CH>(r).  It makes both access
// patterns used by the kernels bank-conflict free: 16 consecutive rows at one logical
// chunk (MFMA row fragments, 16-byte reads) and 4 consecutive rows x 4 consecutive chunks
// (one phase of the transposing 8-byte reads).  swz_f only looks at the low 4 bits of the
// row, so offsets of 16 rows (and of 32-row blocks) fold into immediate offsets.
template <int CH>
__device__ __forceinline__ int swz_f(int row) {
  if constexpr (CH == 16) {
    return ((row & 3) << 2) | ((row >> 2) & 3);
  } else {
    static_assert(CH == 8, "rows of 8 or 16 chunks");
    return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
  }
}
template <int CH>
__device__ __forceinline__ int swz(int row, int chunk) {
  return chunk ^ swz_f<CH>(row);
}
// The swizzle of the kernels built on 16x16x32 MFMAs (A / B: lane = row or column l % 16,
// 8 consecutive k at 8 (l / 16); C: lane = column l % 16, rows 4 (l / 16) + i).  Their access
// patterns: 16 consecutive rows x 4 consecutive chunks (row fragments, 16-byte reads: lane =
// row l % 16, chunk 4 ks + l / 16) and 16 consecutive rows x 2 consecutive chunks (transposing
// 8-byte reads: row 4 (l / 16) + (l % 16) / 4).  The functions are GF(2)-linear in the row and
// were picked by measurement: of all linear maps, run through both patterns on the hardware,
// these are among those that reach the full LDS rate in both (an obvious candidate, the row's
// low three bits shifted up by one with bit 3 as the lowest bit, runs the 16-byte pattern at
// half rate).  They look at the row's low three bits only.
template <int CH>
__device__ __forceinline__ int swz16_f(int row) {
  if constexpr (CH == 16) {
    return ((row & 1) ? 0xc : 0) ^ ((row & 2) ? 0x8 : 0) ^ ((row & 4) ? 0x2 : 0);
  } else {
    static_assert(CH == 8, "rows of 8 or 16 chunks");
    return ((row & 1) ? 0x6 : 0) ^ ((row & 2) ? 0x7 : 0) ^ ((row & 4) ? 0x2 : 0);
  }
}
template <int CH, bool W16>
__device__ __forceinline__ int swz_sel(int row) {
  if constexpr (W16) return swz16_f<CH>(row);
  else return swz_f<CH>(row);
}

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short s16x8;

// Two transposing reads -> one 8-element MFMA fragment.
template <typename V8>
__device__ __forceinline__ V8 tr_pair(const char* p0, const char* p1) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p1);
  const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  V8 out;
  __builtin_memcpy(&out, &both, 16);
  return out;
}

typedef __attribute__((address_space(3))) void lds_void_t;

// Buffer resource over the rows of one (sequence, head) slice: `rows` rows of `row_bytes`
// useful bytes, `stride_bytes` apart.  Loads past the last row return zero, in registers
// and in LDS alike, so partial tiles need no clamping.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rows_rsrc(const void* base, int rows,
                                                                 int64_t stride_bytes,
                                                                 int row_bytes) {
  const int64_t bytes = rows > 0 ? (int64_t)(rows - 1) * stride_bytes + row_bytes : 0;
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
}

// Where the ROWS-row tile that starts at row `row0` of a slice of `rows` rows is fetched from:
// a resource and the byte offset of the tile's first row inside it (rows past the slice's
// last read as zero).
//   FAR = false: the resource covers the whole slice (loop-invariant) and the offset selects the
//                tile; the slice must span less than 2 GiB.
//   FAR = true:  the resource is based at the tile's first row (64-bit pointer arithmetic, all
//                else 32-bit scalar arithmetic) and covers the tile only, so that a slice may
//                span any number of bytes as long as one tile spans less than 2 GiB.  Costs a
//                dozen scalar instructions per tile (2 % of the dK/dV kernel, whose single wave
//                per SIMD hides nothing), which is why the host picks it only when needed.
struct TileSrc {
  __amdgpu_buffer_rsrc_t rsrc;
  int soff;
};
template <int ROWS, bool FAR>
__device__ __forceinline__ TileSrc tile_src(const void* base, int row0, int rows, int stride_bytes,
                                            int row_bytes) {
  if constexpr (FAR) {
    const int n = min(rows - row0, ROWS);  // rows of the tile that exist
    const int bytes = n > 0 ? (n - 1) * stride_bytes + row_bytes : 0;
    const uint64_t off = (uint64_t)(uint32_t)row0 * (uint64_t)(uint32_t)stride_bytes;
    return {__builtin_amdgcn_make_buffer_rsrc((void*)((const char*)base + off), 0, bytes, 0x00020000),
            0};
  } else {
    return {make_rows_rsrc(base, rows, stride_bytes, row_bytes), row0 * stride_bytes};
  }
}

// Key rows in two ranges (AttnArgs::seg): where the tile of key rows starting at `row0` (never straddling the
// boundary: seg is a multiple of every tile size) is fetched from.  What does not depend on the tile is made
// once, 12 scalar instructions a tile less (29 calls: dQ 0.4 % faster, the forward 0.2 %).
template <typename T, int ROW_BYTES, bool FAR>
struct KeyRows {
  const T *first, *second;
  int seg, rows1, rows2;  // boundary; rows of the ranges
  int bytes1, bytes2;     // that they span
  int stride_bytes;
  __device__ __forceinline__ KeyRows(const T* p1, const T* p2, int seg_, int len_k, int64_t stride_elems)
      : first(p1), second(p2), seg(seg_), rows1(min(len_k, seg_)), rows2(len_k - seg_),
        stride_bytes((int)(stride_elems * 2)) {
    bytes1 = rows1 > 0 ? (rows1 - 1) * stride_bytes + ROW_BYTES : 0;
    bytes2 = rows2 > 0 ? (rows2 - 1) * stride_bytes + ROW_BYTES : 0;
  }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t first_range() const {
    return __builtin_amdgcn_make_buffer_rsrc((void*)first, 0, bytes1, 0x00020000);
  }
  template <int ROWS>
  __device__ __forceinline__ TileSrc tile(int row0) const {
    const bool s2 = row0 >= seg;
    const T* base = s2 ? second : first;
    const int row = row0 - (s2 ? seg : 0);
    if constexpr (FAR) {
      return tile_src<ROWS, true>(base, row, s2 ? rows2 : rows1, stride_bytes, ROW_BYTES);
    } else {
      return {__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, s2 ? bytes2 : bytes1, 0x00020000),
              row * stride_bytes};
    }
  }
};

// Cooperative copy of a [ROWS x D] tile into a swizzled LDS tile with buffer loads that
// land directly in LDS (buffer_load_dwordx4 ... lds: lane L of a wave writes
// wave_base + 16 L).  The per-lane byte offsets are computed once (init); a tile load is
// then N instructions with one scalar offset and no vector arithmetic at all.
template <int D, int ROWS, int THREADS, bool W16 = false>
struct TileDma {
  static constexpr int CPR = D / 8;
  static constexpr int RPI = 64 / CPR;  // rows per wave instruction
  static constexpr int NW = THREADS / 64;
  static constexpr int N = ROWS * CPR / THREADS;
  static_assert(N >= 1 && N * THREADS == ROWS * CPR, "tile must divide evenly");
  // Instruction n of a wave covers rows (n NW + wave) RPI + lane / CPR: NW RPI (a multiple
  // of 16) rows further per n, which leaves the swizzle unchanged, so one per-lane offset
  // serves all N instructions and the step goes into the scalar offset.
  static_assert((NW * RPI) % 16 == 0, "row step must preserve the swizzle");
  int voff;
  int step_bytes;
  int wave;
  __device__ __forceinline__ void init(int64_t stride_elems, int tid) {
    const int lane = tid & 63;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = wave * RPI + lane / CPR;
    voff = (int)(row * stride_elems * 2) + (((lane % CPR) ^ swz_sel<CPR, W16>(row)) << 4);
    step_bytes = (int)(NW * RPI * stride_elems * 2);
  }
  // `soff` = byte offset of the tile's first row inside the resource (wave-uniform)
  __device__ __forceinline__ void load_one(__amdgpu_buffer_rsrc_t rsrc, int soff, char* lds_tile,
                                           int n) const {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rsrc, (lds_void_t*)(lds_tile + (n * NW + wave) * 1024), 16, voff, soff + n * step_bytes, 0,
        0);
  }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, int soff, char* lds_tile) const {
#pragma unroll
    for (int n = 0; n < N; n++) load_one(rsrc, soff, lds_tile, n);
  }
  __device__ __forceinline__ void load(const TileSrc& t, char* lds_tile) const {
    load(t.rsrc, t.soff, lds_tile);
  }
};

// The four words of a buffer resource over `bytes` bytes at `base`, for inline assembly.
__device__ __forceinline__ u32x4 rsrc_words(const void* base, int bytes) {
  const uint64_t p = (uint64_t)base;
  return u32x4{(uint32_t)p, (uint32_t)(p >> 32) & 0xffffu, (uint32_t)bytes, 0x00020000u};
}
// tile_src in that form: the resource of the tile whose first row is row0 (FAR: based at that row)
template <int ROWS, bool FAR>
__device__ __forceinline__ u32x4 tile_words(const void* base, int row0, int rows, int stride_bytes,
                                            int row_bytes) {
  if constexpr (FAR) {
    const int n = min(rows - row0, ROWS);
    const uint64_t off = (uint64_t)(uint32_t)row0 * (uint64_t)(uint32_t)stride_bytes;
    return rsrc_words((const char*)base + off, n > 0 ? (n - 1) * stride_bytes + row_bytes : 0);
  } else {
    return rsrc_words(base, (rows - 1) * stride_bytes + row_bytes);
  }
}
// A load that lands in LDS (lane L of the wave: at `lds` + BYTES L) as inline assembly: the
// compiler does not see it write LDS and so never waits for it on its own -- the caller waits
// (wait_dma) before it reads what was loaded.  For tile buffers picked at run time, which the
// compiler cannot tell apart: with the builtin it would wait for the load in flight before every
// LDS read.  The compiler sets m0 and knows of it; its hazard pass does not look inside.  The wait
// state behind the write of m0 is here, but for loads with an OFFSET (bytes, in LDS and in memory alike), for
// which m0 stays as the load without one left it: the build fails where it is written right ahead of one, too.
// (One write of m0 and one wait state for four loads instead of one each: 40 of the short dK/dV form's 630
// instructions a step; us, dK/dV: a pack of 16384 tokens in sequences of 16 to 1024 224 / 217, 4001 rows, window
// 1024, 154 / 150, 14 drawn calls 2.7 % on average.)  The five between a vector instruction's write of a scalar
// register (what a spilled one comes back by) and its use by the load are not (they cost the short
// dK/dV form 2.8 % over 119 shapes): the build fails where one comes closer (build.py).
template <int BYTES, int OFFSET = 0>
__device__ __forceinline__ void lds_load_asm(u32x4 rsrc, int voff, int soff, uint32_t lds) {
  static_assert(BYTES == 4 || BYTES == 16, "one dword or four per lane");
  if constexpr (BYTES == 16 && OFFSET == 0) {
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :: "v"(voff), "s"(rsrc), "s"(soff), "{m0}"(lds) : "memory");
  } else if constexpr (BYTES == 16) {
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen offset:%4 lds"
                 :: "v"(voff), "s"(rsrc), "s"(soff), "{m0}"(lds), "n"(OFFSET) : "memory");
  } else {
    asm volatile("s_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds"
                 :: "v"(voff), "s"(rsrc), "s"(soff), "{m0}"(lds) : "memory");
  }
}

// TileDma for a tile that one wave loads for itself (layout as of TileDma with swz_f): instruction n
// covers rows n RPI .. n RPI + RPI - 1, fewer than the 16 after which the swizzle repeats, so the
// chunk part of the lane offset takes one of 16 / RPI forms in turn, made by one XOR-and-add from
// the lane's chunk in the tile's first rows (`chunk`, the same for every tensor).
template <int D, int ROWS>
struct WaveTileDma {
  static constexpr int CPR = D / 8;
  static constexpr int RPI = 64 / CPR;
  static constexpr int N = ROWS * CPR / 64;
  int row_off;
  int step_bytes;
  static __device__ __forceinline__ int chunk(int lane) {
    return ((lane % CPR) ^ swz_f<CPR>(lane / CPR)) << 4;
  }
  __device__ __forceinline__ void init(int64_t stride_elems, int tid) {
    row_off = (int)((tid & 63) / CPR * stride_elems * 2);
    step_bytes = (int)(RPI * stride_elems * 2);
  }
  // `rsrc`: of the rows and the BACK bytes ahead of them, which no lane reads; `soff` is the tile's place among the
  // rows.  What sharing a write of m0 takes out of the scalar offset, an unsigned number, can leave none below zero
  // so, also where rows lie closer than their own bytes (the gradient of a sum over the rows: stride 0).
  static constexpr int BACK = 3 * 1024;
  template <int NTH>
  __device__ __forceinline__ void load_one(u32x4 rsrc, int soff, uint32_t lds_tile, int chunk0) const {
    // rows n RPI + r, r < RPI: swz_f(n RPI + r) = swz_f(r) ^ swz_f(n RPI)
    constexpr int x = (CPR == 16 ? NTH & 3 : (NTH & 1) << 1) << 4;
    constexpr int at = (NTH & 3) * 1024;  // (the instruction's offset counts in LDS and in memory)
    static_assert(at <= BACK, "no scalar offset below zero");
    lds_load_asm<16, at>(rsrc, (chunk0 ^ x) + row_off, soff + NTH * step_bytes - at, lds_tile + NTH * 1024 - at);
  }
};

// f(integral_constant<int, 0>{}), ..., f(integral_constant<int, N - 1>{}): a loop whose
// index is a compile-time constant in every iteration (register arrays indexed by it never
// fall back to dynamic indexing, whatever the unroller thinks of the body's size).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// put(i, visible(i)) for i = 0 .. N - 1, compile-time constants, the comparisons (visible: a mask of lanes) of
// four ahead of their selects: a select right behind its comparison waits two states for the lane mask, 32 times
// in an edge tile.  (us, before / after: forward of 2 x 333 rows, 8 / 2 heads, window 100, fp16, 10.0 / 9.7;
// 24 drawn and listed calls, forward 2.0 % on average, dK/dV 0.9 %.  The dQ kernel keeps
// plain selects: it has no scalar registers for this, 96 become 142 spilled and the rank step's dQ 683 / 708.)
__device__ __forceinline__ uint64_t lanes(bool x) { return __builtin_amdgcn_ballot_w64(x); }
template <int N, typename Visible, typename Put>
__device__ __forceinline__ void select_lanes(Visible&& visible, Put&& put) {
  static_assert(N % 4 == 0, "four at a time");
  static_for<N / 4>([&](auto bc) __attribute__((always_inline)) {
    constexpr int i = 4 * decltype(bc)::value;
    uint64_t m[4];
    static_for<4>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      m[j] = visible(std::integral_constant<int, i + j>{});
    });
    asm volatile("" : "+s"(m[0]), "+s"(m[1]), "+s"(m[2]), "+s"(m[3]));
    static_for<4>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      put(std::integral_constant<int, i + j>{}, __builtin_amdgcn_inverse_ballot_w64(m[j]));
    });
  });
}

// Block barrier that waits for this wave's LDS traffic only: loads still in flight from
// global memory into LDS (vmcnt) are NOT drained, unlike __syncthreads().  A wave that
// issued such loads calls wait_dma() before the barrier that publishes them.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_dma() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Wait until at most N of this wave's vector memory operations (loads, loads into LDS, stores:
// they complete in issue order) are outstanding.  Through the builtin, so that the compiler's own
// bookkeeping of what is in flight sees the wait (gfx9 encoding: vmcnt in bits 3:0 and 15:14,
// the other counters left at their "no wait" values).
template <int N>
__device__ __forceinline__ void wait_vmem_but() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
}

// max / sum across the two half-waves (lane l <-> lane l ^ 32).
__device__ __forceinline__ float halfwave_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halfwave_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Keys per block of the dK/dV kernel
constexpr int kDkvKeysPerBlock = 256;
// dS hand-off: bytes one dK/dV block leaves per 32-row query tile (32 x 256 16-bit values) and
// per wave of it (32 x 64: the unit the dQ kernel of that route fetches)
constexpr int kDsBlockBytes = 32 * kDkvKeysPerBlock * 2;
constexpr int kDsUnitBytes = kDsBlockBytes / 4;
constexpr int kMaxTileRows = 256;  // bound on the rows fetched as one tile that the stride checks assume
                                   // (today's largest tile has 64 rows: K / V in the forward and dQ kernels)
struct BwdLayout {
  uint64_t stats_bytes;    // each of the two statistics arrays
  int n_count;             // arrival counters of the sink kernel
  uint64_t count_off, total_bytes;
  uint64_t ktile_off;      // key tile table of a pack (0: none)
  int sink_chunks;         // row chunks of the sink kernel per (sequence, kv head); 0: no sink kernel
  uint64_t sink_off;       // its fp32 sums
  // dS hand-off (ds_bytes == 0: not used for this call)
  uint64_t ds_off, ds_bytes;
  int ds_nkb, ds_slots;
};
// (`max_bytes`: room there is; where the whole would not fit, the key tile table of a pack is left out, which
// only costs time, and where that is not enough the sink kernel gets fewer chunks: the same sums in another
// order)
BwdLayout bwd_layout(const rswa_attn_params* p, bool allow_handoff, uint64_t max_bytes = ~0ull);

// Fill an AttnArgs from the public struct; validates what both directions share.
int fill_args(const rswa_attn_params* p, bool backward, AttnArgs& a, bool allow_handoff = false,
              uint64_t max_bytes = ~0ull);

}  // namespace rswa
