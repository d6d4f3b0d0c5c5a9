// Band / sink attention backward for gfx950, without atomics.
//
// Replaces flash-attn's backward as wrapped at ring_swa/ops/wrap_flash.py:276-429.
// Launches on the caller's stream: DQ (which makes the row statistics, too), then DKDV; for packs
// and sink keys a one-block kernel ahead of them.  Where the phases are asked for in separate calls,
// or DQ cannot make the statistics, PREP, then DKDV and DQ:
//   PREP : per (row, q head): -delta = -sum_d dO * O and -lse2 = -lse * log2(e) (stored negated:
//          they enter the kernels as addends),
//          both fp32, into the caller's workspace
//   DKDV : one block (4 waves, one per SIMD, up to 512 registers each) owns 256 keys of one
//          (sequence, kv head) and walks the query tiles (32 rows) that can see them, for
//          every q head of the GQA group; a wave owns 64 keys: their K and V fragments stay
//          in registers, dK^T / dV^T accumulate in accumulation registers for the whole
//          walk and are written once.  Where such blocks would leave compute units idle a
//          block owns 64 keys instead and its waves share out the walk (WALK4)
//   DQ   : one block (8 waves x 32 query rows: 128 rows of two q heads of a GQA group, or
//          256 rows of one head) walks the key tiles (64 keys) it can see, like the forward
//          kernel; dQ^T stays in registers
// S and dP are computed in both main kernels (7 GEMM units instead of 5).  That costs
// less here than fp32 atomics on dQ: hardware fp32 atomic adds retire at 340 G elements/s on
// the whole device (measured with 64 consecutive floats per wave instruction, the pattern a
// fused kernel would use), a dQ tile of 32 x 128 per 256-key block and step needs 700 G/s at
// the rate the dK/dV kernel walks.  It also makes the result run-to-run deterministic.
//
// DKDV per (query tile, wave) (C layout: lane = key; two 32-key blocks per wave, so every
// fragment read from LDS feeds two MFMAs):
//   S = Q K^T, dP = dO V^T      A = Q / dO row fragments (LDS), B = K / V (registers)
//   P = exp2(S*c - lse2), dS = P * (dP - delta); the dP chains start from -delta instead of zero.
//   (Folding c into 16-bit K fragments and starting the S chains from -lse2 would save the
//   multiply-add per score -- 1-2 % -- but the rounding of K c shifts the exponent by up to
//   2^-9 |S c|: with peaked scores, e.g. sink keys four times the usual size, it doubled the
//   error of dK / dV against the fp32 oracle, 4e-3 -> 7e-3.  The scale stays in fp32.)
//   dV^T += dO^T P, dK^T += Q^T dS   A = transposing LDS reads of dO / Q, B = P / dS (regs)
// The S and dP MFMAs are inline assembly so that their accumulators live in vector
// registers, where the vector ALU reads them next; left to the compiler they end up in
// accumulation registers like dK^T and dV^T and every element costs two copies.  The
// compiler does not know that these statements are MFMAs and pads nothing after them:
// the code keeps at least two later MFMAs between the last one that writes S or dP and
// the first read of the result.  The dK^T / dV^T MFMAs are compiler builtins (accumulation
// registers), so every copy or read the compiler adds around them is padded as required.
// DQ per (key tile, wave), on 16x16x32 MFMAs; wave owns 32 query columns (lane = query l % 16
// of two 16-query blocks):
//   S^T = K Q^T, dP^T = V dO^T  A = K / V row fragments from LDS, B = Q / dO fragments (regs);
//                               the dP^T chains start from -delta of the lane's queries
//   dS^T = exp2(S^T c - lse2) dP^T   (the scale is applied in fp32: see the note at DKDV)
//   dQ^T += K^T dS^T            A = transposing LDS reads of K, B = dS^T (regs)
//
// Streamed tiles are double-buffered in SEPARATE static __shared__ arrays, filled by buffer
// loads that land directly in LDS one tile ahead, and the tile loops are unrolled by two so
// that every access names its buffer statically (see attn_fwd.hip for why).
#include "attn_common.h"

#include <algorithm>
#include <cmath>
#include <mutex>

namespace rswa {
namespace {

// One lane's 8 consecutive values of a gradient row, already rounded to the 16-bit type, into
// the caller's buffer at element offset `at`: as they are, as fp32 (a ring accumulator), and in
// either case added to what the buffer holds (fp32 sum, one rounding for a 16-bit buffer).
template <typename T>
__device__ __forceinline__ void put_grad8(void* buf, int64_t at, typename Mma<T>::V8 val, bool wide,
                                          bool accumulate) {
  using V8 = typename Mma<T>::V8;
  if (wide) {
    float* dst = (float*)buf + at;
    f32x4 y[2];
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
      f32x4 old = {0.f, 0.f, 0.f, 0.f};
      if (accumulate) old = *(const f32x4*)(dst + 4 * hh);
#pragma unroll
      for (int j = 0; j < 4; j++) y[hh][j] = old[j] + (float)val[4 * hh + j];
    }
    *(f32x4*)dst = y[0];
    *(f32x4*)(dst + 4) = y[1];
  } else {
    T* dst = (T*)buf + at;
    if (accumulate) {
      const V8 old = *(const V8*)dst;
      float sum[8];
#pragma unroll
      for (int j = 0; j < 8; j++) sum[j] = (float)old[j] + (float)val[j];
      val = Mma<T>::pack(sum);
    }
    *(V8*)dst = val;
  }
}

// N times a wave's rows of a gradient tile, RPI rows each: get(n) is the lane's 8 values of its row
// n RPI, at element offset `at` + n RPI row_st of the buffer; of its rows the lane owns those with
// n RPI < left (all of them where `all`, a uniform condition, says so).
template <typename T, int RPI, int N, typename Get>
__device__ __forceinline__ void put_rows(void* buf, int64_t at, int64_t row_st, int left, bool all, bool wide,
                                         bool accumulate, Get&& get) {
  using V8 = typename Mma<T>::V8;
  const int64_t step = RPI * row_st;
  if (!(wide | accumulate)) {
    T* dst = (T*)buf + at;
    if (all) {
#pragma unroll
      for (int n = 0; n < N; n++) *(V8*)(dst + n * step) = get(n);
    } else {
#pragma unroll
      for (int n = 0; n < N; n++)
        if (n * RPI < left) *(V8*)(dst + n * step) = get(n);
    }
  } else {
#pragma unroll 1
    for (int n = 0; n < N; n++)
      if (n * RPI < left) put_grad8<T>(buf, at + n * step, get(n), wide, accumulate);
  }
}

// Sequences of at most this many keys whose dK/dV blocks take the snake order (see the kernel)
constexpr int kSnakeKeys = 4096;

// ============================================================================
// dK / dV
// ============================================================================
// rows of a query tile of the dK/dV kernel, whose statistics it reads together
constexpr int kStatTileRows = 32;

template <int D>
struct DkvCfg {
  static constexpr int BM = kStatTileRows;  // query rows per step
  static constexpr int KB = 2;         // 32-key blocks per wave
  static constexpr int BN = kDkvKeysPerBlock;  // keys per block: 4 waves x KB x 32
  static_assert(BN == 256, "4 waves x KB x 32 keys");
  static constexpr int THREADS = 256;  // one wave per SIMD, up to 512 registers each
  static constexpr int KSTEPS = D / 16;
  static constexpr int DBLK = D / 32;
  static constexpr int CPR = D / 8;   // 16-byte chunks per row
  static constexpr int ROWB = D * 2;  // bytes per row
  static constexpr int Q_TILE = BM * ROWB;
};

// WALK4: the block owns 64 keys, all four waves hold the same K and V fragments and take turns on
// the walk (q heads dealt to the waves; with fewer than four in the group also query tiles), each
// fetching its own Q / dO tiles into its own buffers -- no barrier in the walk, and a wave's keys
// are the block's, so no step is idle for some waves.  The four partial sums are added in LDS at
// the end, in wave order.  Four times as many, four times as short blocks for launches that would
// otherwise fill the chip badly (small launches, short sequences, sizes just above a full round),
// a longer tile fetch per step (four tiles instead of one shared), so blocks that fill the chip by
// themselves stay wide: see dkv_walk4.  It took the place of blocks of 256 keys whose q heads were
// split over 2-4 blocks with fp32 partial sums in memory: us, dK/dV alone, bf16, head_dim 128, 32 / 8
// heads: window 1024, 4001 rows 180 -> 127; full causal attention over 2048 / 4096 rows 111 -> 98 / 261
// -> 244; 28 / 4 heads (which could not be split evenly), 2000 rows, 368 -> 97.
template <typename T, int D, bool FAR, bool HAND, bool WALK4>
__global__ __launch_bounds__(256) void attn_bwd_dkdv_kernel(const AttnArgs a) {
  static_assert(!(HAND && FAR), "dS hand-off in the first addressing form only");
  using C = DkvCfg<D>;
  constexpr int BN = WALK4 ? C::BN / 4 : C::BN;  // keys of the block
  using M = Mma<T>;
  using V8 = typename M::V8;
  constexpr int KB = C::KB, KS = C::KSTEPS, DB = C::DBLK;
  // (WALK4: q_s0 holds every wave's own four tile buffers, wave after wave, the st_* every wave's
  // own statistics)
  constexpr int W_LDS = 4 * C::Q_TILE;  // LDS bytes of one wave's tile buffers
  __shared__ __attribute__((aligned(1024))) char q_s0[WALK4 ? 4 * W_LDS : C::Q_TILE];
  __shared__ __attribute__((aligned(1024))) char q_s1[WALK4 ? 16 : C::Q_TILE];
  __shared__ __attribute__((aligned(1024))) char do_s0[WALK4 ? 16 : C::Q_TILE];
  __shared__ __attribute__((aligned(1024))) char do_s1[WALK4 ? 16 : C::Q_TILE];
  __shared__ __attribute__((aligned(1024))) float st_s0[(WALK4 ? 8 : 2) * C::BM];  // -lse2[BM], -delta[BM]
  __shared__ __attribute__((aligned(1024))) float st_s1[(WALK4 ? 8 : 2) * C::BM];

  // A pack's exact number of key tiles is known on the device only (ktile, see
  // write_ktile): the tiles come first in the launch, dealt evenly to the XCDs, and the blocks beyond
  // them end here.  Consecutive blocks of an XCD go to its shader engines in turn and wait for the
  // engine whose turn it is, so lengths that repeat with an even period leave engines idle: with a
  // pack's tiles numbered by slots, one of them unused per sequence, as in the other kernels, 64
  // sequences of 256 tokens (32 / 8 heads, head_dim 128) took 242 us, every other block being empty;
  // numbered exactly, 129 us.  `snake` reverses every other group of four blocks where the walks
  // of a sequence's few tiles are such a pattern: of 256-key tiles only a number that is a multiple
  // of four repeats in step with the engines (us, plain / snake, all alike: 64 sequences of 1024
  // tokens, 32 / 32 heads, 1720 / 1400; dense causal, head_dim 64, 4016 rows x 32 heads 188 / 170; but
  // 1954 rows against 2466 keys, ten tiles, 59 / 67, 2 x 1110 rows, five, 54 / 61), of the 64-key
  // form's tiles any (422 shapes, mean 1.2 % faster, 10 % slower to 20 % faster).  Sequences of
  // more than 4096 keys keep the plain order: four of 16384 tokens lose 3 % by it, 10240 keys under
  // 8192 rows in 40 wide tiles 447 / 550.
  // (which tiles an XCD takes: see tile_of_block)
  int n_tile = a.n_tile, n_group = a.n_group, snake = a.snake;
  if (a.ktile) {
    n_tile = a.ktile[a.batch];
    snake = a.ktile[a.batch + 1];
    n_group = n_tile * (a.heads_kv << a.xcd_log2 >> 3);
  }
  const int xcd = (int)blockIdx.x & 7, in_group = (1 << a.xcd_log2) - 1;
  int per_xcd = (n_group + in_group) >> a.xcd_log2;
  if (a.xcd_log2 == 0) per_xcd = (n_tile * a.tile_heads + 7) >> 3;
  int in_xcd = (int)blockIdx.x >> 3;
  if (in_xcd >= per_xcd) return;
  if (snake && (in_xcd & 4) && (in_xcd | 3) < per_xcd) in_xcd ^= 3;
  int wid = xcd * per_xcd + in_xcd;
  if (a.xcd_log2 == 0) {
    if (wid >= n_tile * a.tile_heads) return;
  } else {
    const int at_group = (in_xcd << a.xcd_log2) + (xcd & in_group);
    if (at_group >= n_group) return;
    wid = (xcd >> a.xcd_log2) * n_group + at_group;
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (not WALK4: key group of 64 keys)
  const int l32 = lane & 31;
  const int g = lane >> 5;
  const int i16 = lane & 15;
  const int u = lane >> 4;

  // ---- which (sequence, kv head, key tile); tiles go heaviest first -------------------
  const int slot = a.rev_k ? n_tile - 1 - wid % n_tile : wid % n_tile;
  int rest = wid / n_tile;
  const int hk = rest % a.heads_kv;
  SeqInfo s;
  int kt;
  if (a.ktile) {
    locate_tile(a, slot, s, kt);
  } else if (a.cu_q) {
    static_assert(C::BN == 1 << 8, "tile size passed to locate_packed");
    if (!locate_packed(a, slot, WALK4 ? 6 : 8, true, s, kt)) return;
  } else {
    s.batch_idx = rest / a.heads_kv;
    s.q_row0 = s.k_row0 = 0;
    s.len_q = a.seqlen_q;
    s.len_k = a.seqlen_k;
    kt = slot;
  }
  const int b = s.batch_idx;
  const int len_q = s.len_q, len_k = s.len_k;
  const int j0 = kt * BN;
  if (j0 >= len_k) return;
  const int j_last = min(j0 + BN, len_k) - 1;
  const int shift = a.shift_explicit ? a.shift_val : len_k - len_q;

  // Keys in two row ranges (dense mode; the boundary is a multiple of the block's keys): the
  // block's keys all lie in one of them, and its pointers are set so that a key's index in the
  // sequence selects its row.
  const bool seg2 = j0 >= a.seg;
  const int64_t seg_row0 = seg2 ? -(int64_t)a.seg : s.k_row0;
  const T* k_ptr = (const T*)(seg2 ? a.k2 : a.k) + b * a.k_st[0] + seg_row0 * a.k_st[1] + hk * a.k_st[2];
  const T* v_ptr = (const T*)(seg2 ? a.v2 : a.v) + b * a.v_st[0] + seg_row0 * a.v_st[1] + hk * a.v_st[2];
  // (gradient buffers: T or, as ring accumulators, fp32 -- element offsets)
  void* const dk_buf = seg2 ? a.dk2 : a.dk;
  void* const dv_buf = seg2 ? a.dv2 : a.dv;
  const int64_t dk_off = b * a.dk_st[0] + seg_row0 * a.dk_st[1] + hk * a.dk_st[2];
  const int64_t dv_off = b * a.dv_st[0] + seg_row0 * a.dv_st[1] + hk * a.dv_st[2];
  const int64_t ws_row0 = a.cu_q ? s.q_row0 : (int64_t)b * a.seqlen_q;

  // ---- query tiles that can see this key tile -------------------------------
  const int i_min = (a.wr >= 0) ? max(0, j0 - shift - a.wr) : 0;
  const int i_max =
      (a.wl >= 0) ? min(len_q - 1, j_last - shift + a.wl) : len_q - 1;
  const int qt_lo = i_min / C::BM;
  const int n_qt = (i_max >= i_min) ? i_max / C::BM - qt_lo + 1 : 0;
  // WALK4: the walk is dealt to the waves, 1 << hw_log2 q heads at a time and, of a head's query
  // tiles, every (1 << tw_log2)-th to each wave on it
  const int hw_log2 = WALK4 ? ((a.group & 3) == 0 ? 2 : (a.group & 1) == 0 ? 1 : 0) : 0;
  const int tw_log2 = WALK4 ? 2 - hw_log2 : 0;
  const int w_tile = WALK4 ? wave >> hw_log2 : 0;  // the wave's first tile of a head's walk
  const int w_tiles = (n_qt - w_tile + (1 << tw_log2) - 1) >> tw_log2;
  const int n_iter = WALK4 ? w_tiles * (a.group >> hw_log2) : n_qt * a.group;

  const int jw0 = WALK4 ? j0 : j0 + wave * (32 * KB);  // first key column of this wave
  const int jw1 = jw0 + 32 * KB - 1;

  // ---- lane-constant LDS offsets (swizzle folded: varying parts are XOR / immediates) ----
  // 16-byte row fragments: row = l32 (+ 32 per block), chunk = 2 ks + g
  //   offset = (a_row ^ (ks << 5)) + blk * 32 * ROWB
  const int w_lds = WALK4 ? wave * W_LDS : 0;  // (a multiple of what the XORs touch)
  const int a_row = w_lds + l32 * C::ROWB + ((g ^ swz_f<C::CPR>(l32)) << 4);
  // transposing reads of Q / dO: rows 16 ks + 4 g + (i16 >> 2) and + 8, chunk = 4 d + lp
  //   offset = (t_row{0,1} ^ (d << 6)) + ks * 16 * ROWB
  const int rl = 4 * g + (i16 >> 2);
  const int lp = 2 * (u & 1) + ((i16 & 3) >> 1);
  const int t_row0 = w_lds + rl * C::ROWB + ((lp ^ swz_f<C::CPR>(rl)) << 4) + (i16 & 1) * 8;
  const int t_row1 = w_lds + (rl + 8) * C::ROWB + ((lp ^ swz_f<C::CPR>(rl + 8)) << 4) + (i16 & 1) * 8;

  // ---- this wave's K fragments stay in registers for the whole walk (B operand of
  // S = Q K^T: lane = key column, 8 consecutive d per k-step)
  // (keys past the end read the last one's values: their columns are masked in every tile and never
  // stored)
  V8 kf[KB][KS], vf[KB][KS];  // (the V fragments: B operand of dP = dO V^T, same layout)
  // WALK4: all four waves want the same 64 rows, which come through LDS, where the tiles of odd steps will
  // be: a wave's direct loads touch 32 rows with 32 bytes each, and a block's 128 of them took its vector
  // memory unit 2 of the block's first 5 us (us, dK/dV, direct / staged: 4001 rows, window 1024, 32 / 8 heads
  // 125 / 121; a pack of 16384 tokens in sequences of 16 to 1024 220 / 208)
  [[maybe_unused]] char *const k_stage = q_s0 + 2 * C::Q_TILE, *const v_stage = q_s0 + (WALK4 ? W_LDS : 0) + 2 * C::Q_TILE;
  if constexpr (WALK4) {
    const int rows = min(len_k - j0, 64);
    const auto stage_rows = [&](const T* base, int64_t st, char* dst) __attribute__((always_inline)) {
      TileDma<D, 64, 256> dma;
      dma.init(st, tid);
      dma.load(make_rows_rsrc(base + (int64_t)j0 * st, rows, st * 2, C::ROWB), 0, dst);  // (rows past the end: zero)
    };
    stage_rows(k_ptr, a.k_st[1], k_stage);
    stage_rows(v_ptr, a.v_st[1], v_stage);
  } else {
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      const int jc = min(jw0 + kb * 32 + l32, len_k - 1);
      const T* k_row = k_ptr + (int64_t)jc * a.k_st[1] + g * 8;
      const T* v_row = v_ptr + (int64_t)jc * a.v_st[1] + g * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) kf[kb][ks] = *(const V8*)(k_row + ks * 16);
#pragma unroll
      for (int ks = 0; ks < KS; ks++) vf[kb][ks] = *(const V8*)(v_row + ks * 16);
    }
  }
  f32x16 dk_acc[KB][DB], dv_acc[KB][DB];
#pragma unroll
  for (int kb = 0; kb < KB; kb++)
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        dk_acc[kb][d][i] = 0.f;
        dv_acc[kb][d][i] = 0.f;
      }
  if constexpr (WALK4) {
    // (opaque zeros: the compiler takes a loop-carried vector that starts from a constant apart into
    // scalars, which live in vector registers and are copied to accumulation registers every step)
#pragma unroll
    for (int kb = 0; kb < KB; kb++)
#pragma unroll
      for (int d = 0; d < DB; d++) asm volatile("" : "+a"(dk_acc[kb][d]), "+a"(dv_acc[kb][d]));
  }
  // ---- tile DMA (rows past the end of the sequence read as zero) ------------------
  using Dma = std::conditional_t<WALK4, WaveTileDma<D, C::BM>, TileDma<D, C::BM, C::THREADS>>;
  Dma q_dma, do_dma;
  q_dma.init(a.q_st[1], tid);
  do_dma.init(a.do_st[1], tid);
  constexpr int BACK = WALK4 ? WaveTileDma<D, C::BM>::BACK : 0;  // bytes; see there
  const T* q_base = (const T*)((const char*)a.q - BACK) + b * a.q_st[0] + s.q_row0 * a.q_st[1];
  const T* do_base = (const T*)((const char*)a.dout - BACK) + b * a.do_st[0] + s.q_row0 * a.do_st[1];
  // statistics: one load covers both workspace arrays (lse2, then delta `stat_elems` further
  // on) through one resource, the tile's first row in the scalar offset; rows past the sequence end read
  // a neighbour's finite values, which the row mask / zero Q, dO rows void
  // (element counts below 2^30: the host refuses larger statistics arrays)
  const int stat_elems = (int)(a.delta - a.lse2);  // elements between the two arrays
  const int stat_end = stat_elems + a.heads_q * (int)a.rows_q;  // end of delta
  const int q_row_bytes = (int)(a.q_st[1] * 2), do_row_bytes = (int)(a.do_st[1] * 2);
  // Cursor over the (q head of the group, query tile) pairs, advanced incrementally so
  // that a step costs a handful of scalar instructions: the tile's first row, the head's
  // Q / dO base pointers and the offset of its statistics.  (A lone wave per SIMD pays for each: without a
  // resource of the statistics for every tile (ten, in the wave that the others wait for), a tile count beside
  // the row, a test for the last tile and pairs of comparisons where one will do, 66 scalar instructions a
  // step became 48; dK/dV of 65536 tokens, window 4092, 6664 / 6527 us, of 2 x 8192 rows, 32 heads, window
  // 1000, 620 / 607, the rank step with 14336 keys 1194 / 1162.)
  struct Cursor {
    int qt, i0;
    const T *q_head, *do_head;
    int stat_row;  // index of row 0 of this head in the statistics arrays
    int ds;        // HAND: byte offset of this wave's dS unit of the tile (from ds_first)
  };
  const int i_first = qt_lo * C::BM;
  // Every head's walk over the n_qt query tiles starts at tile qt_start and wraps around,
  // chosen so that at any step all blocks of a kv head whose walks are equally long are
  // on the same query tile modulo n_qt: neighbouring key tiles see almost the same query
  // rows, and walking them in step lets one L2 fill serve all of them.
  const int qt_start = n_qt > 0 ? (n_qt - qt_lo % n_qt) % n_qt : 0;
  Cursor nxt;  // the tile that the load parts fetch
  nxt.qt = w_tile;  // WALK4: position in the walk, counted from qt_start
  auto row_of = [&](int pos) __attribute__((always_inline)) {
    const int at = qt_start + pos;
    return i_first + (at >= n_qt ? at - n_qt : at) * C::BM;
  };
  nxt.i0 = row_of(w_tile);
  // (not WALK4: a head's walk ends behind the last tile at i_end and is through when it is back at i_start)
  const int i_end = i_first + n_qt * C::BM, i_start = nxt.i0;
  int heads_left = a.group - 1;  // heads of the walk after nxt's
  const int h_first = hk * a.group + (WALK4 ? wave & ((1 << hw_log2) - 1) : 0);
  nxt.q_head = q_base + (int64_t)h_first * a.q_st[2];
  nxt.do_head = do_base + (int64_t)h_first * a.do_st[2];
  nxt.stat_row = (int)(h_first * a.rows_q + ws_row0);
  const __amdgpu_buffer_rsrc_t st_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.lse2, 0, (int)((uint32_t)stat_end * 4u), 0x00020000);
  // dS hand-off: unit of (q head h, row tile qt of the sequence, this block's keys, this wave) at
  //   ds + (((h ds_slots + slot0 + qt) ds_nkb + kt % ds_nkb) 4 + wave) 4 KiB
  // -- per step one row of ds_nkb blocks further, per head ds_slots rows further.  The units
  // of the block's heads are addressed as 32-bit offsets from that of its first head's first
  // tile, through a buffer resource that ends with the last head's rows: an offset beyond it
  // (kDsNowhere) makes the hardware drop the store.
  const int ds_row_bytes = HAND ? a.ds_nkb * kDsBlockBytes : 0;
  const int ds_head_bytes = HAND ? a.ds_slots * ds_row_bytes : 0;  // (host: group x this < 2 GiB)
  constexpr int kDsNowhere = 0x7ff00000;
  const int64_t ds_slot0 = a.cu_q ? (s.q_row0 >> 5) + b : (int64_t)b * ((a.seqlen_q + 31) >> 5);
  const int64_t ds_first = HAND ? (int64_t)h_first * ds_head_bytes + (ds_slot0 + qt_lo) * ds_row_bytes +
                                      ((jw0 >> 8) % max(a.ds_nkb, 1)) * kDsBlockBytes +
                                      ((jw0 >> 6) & 3) * kDsUnitBytes
                                : 0;
  const __amdgpu_buffer_rsrc_t ds_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      a.ds + ds_first, 0,
      HAND ? (int)min((int64_t)a.group * ds_head_bytes, (int64_t)a.heads_q * ds_head_bytes - ds_first) : 0,
      0x00020000);
  int ds_head_off = 0;  // of the head the cursor is on
  nxt.ds = ((nxt.i0 - i_first) >> 5) * ds_row_bytes;
  [[maybe_unused]] int cur_ds = nxt.ds;  // the unit of the tile being computed
  // The next tile is fetched by NPART instructions per wave (statistics, Q, dO), issued
  // one at a time between the first MFMAs of a step; advance() then moves the cursor on.
  constexpr int NQD = Dma::N;
  constexpr int NPART = 1 + 2 * NQD;
  const int st_voff = ((lane & 31) << 2) + (lane >> 5) * (stat_elems * 4);
  [[maybe_unused]] int dma_chunk = 0;  // WALK4: see WaveTileDma
  if constexpr (WALK4) dma_chunk = Dma::chunk(lane);
  auto load_part = [&](auto part_c, char* qd, char* dod, float* std_) __attribute__((always_inline)) {
    constexpr int part = decltype(part_c)::value;
    if constexpr (part == 0) {
      if (WALK4 || wave == 0) {  // lanes 0-31: lse2 of the 32 rows, lanes 32-63: their delta
        const int first = nxt.stat_row + nxt.i0;
        if constexpr (WALK4) {
          lds_load_asm<4>(rsrc_words(a.lse2, (int)((uint32_t)stat_end * 4u)), st_voff, first * 4,
                          (uint32_t)(uintptr_t)(lds_void_t*)std_);
        } else {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(st_rsrc, (lds_void_t*)std_, 4, st_voff, first * 4, 0, 0);
        }
      }
    } else if constexpr (WALK4) {
      constexpr bool is_q = part <= NQD;
      const T* head = is_q ? nxt.q_head : nxt.do_head;
      const int row_bytes = is_q ? q_row_bytes : do_row_bytes;
      (is_q ? q_dma : do_dma)
          .template load_one<is_q ? part - 1 : part - 1 - NQD>(
              tile_words<C::BM, FAR>(head, nxt.i0, len_q, row_bytes, C::ROWB + BACK), FAR ? BACK : nxt.i0 * row_bytes + BACK,
              (uint32_t)(uintptr_t)(lds_void_t*)(is_q ? qd : dod) + w_lds, dma_chunk);
    } else if constexpr (part <= NQD) {
      const TileSrc t = tile_src<C::BM, FAR>(nxt.q_head, nxt.i0, len_q, q_row_bytes, C::ROWB);
      q_dma.load_one(t.rsrc, t.soff, qd, part - 1);
    } else {
      const TileSrc t = tile_src<C::BM, FAR>(nxt.do_head, nxt.i0, len_q, do_row_bytes, C::ROWB);
      do_dma.load_one(t.rsrc, t.soff, dod, part - 1 - NQD);
    }
  };
  // may the cursor be advanced beyond the last tile?  (with the dS hand-off the kernel spills without the test)
  constexpr bool FREE_RUN = !WALK4 && !HAND;
  auto advance = [&]() __attribute__((always_inline)) {
    if constexpr (WALK4) {
      nxt.qt += 1 << tw_log2;
      if (nxt.qt >= n_qt) {
        nxt.qt = w_tile;
        nxt.q_head += a.q_st[2] << hw_log2;
        nxt.do_head += a.do_st[2] << hw_log2;
        nxt.stat_row += (int)a.rows_q << hw_log2;
        if constexpr (HAND) ds_head_off += ds_head_bytes << hw_log2;
      }
      nxt.i0 = row_of(nxt.qt);
      if constexpr (HAND) nxt.ds = ds_head_off + ((nxt.i0 - i_first) >> 5) * ds_row_bytes;
      return;
    }
    // (past the last head's walk the cursor stays on that head: its tiles are fetched again, into buffers
    // nobody reads)
    nxt.i0 += C::BM;
    if constexpr (HAND) nxt.ds = nxt.i0 == i_end ? ds_head_off : nxt.ds + ds_row_bytes;
    nxt.i0 = nxt.i0 == i_end ? i_first : nxt.i0;
    if (nxt.i0 == i_start && heads_left > 0) {
      heads_left--;
      nxt.q_head += a.q_st[2];
      nxt.do_head += a.do_st[2];
      nxt.stat_row += (int)a.rows_q;
      if constexpr (HAND) {
        ds_head_off += ds_head_bytes;
        nxt.ds += ds_head_bytes;
      }
    }
  };

  // buffers of the even and odd steps
  char *const qb0 = q_s0, *const qb1 = WALK4 ? q_s0 + 2 * C::Q_TILE : q_s1;
  char *const dob0 = WALK4 ? q_s0 + C::Q_TILE : do_s0, *const dob1 = WALK4 ? q_s0 + 3 * C::Q_TILE : do_s1;
  float *const stb0 = WALK4 ? st_s0 + wave * 2 * C::BM : st_s0, *const stb1 = WALK4 ? st_s1 + wave * 2 * C::BM : st_s1;
  int cur_i0 = nxt.i0;  // first row of the tile being computed
  if (n_iter > 0) {
    static_for<NPART>([&](auto pc) __attribute__((always_inline)) { load_part(pc, qb0, dob0, stb0); });
    if (FREE_RUN || n_iter > 1) advance();
  }
  if constexpr (WALK4) {
    wait_vmem_but<0>();
    lds_barrier();
#pragma unroll
    for (int kb = 0; kb < KB; kb++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        const int at = ((a_row - w_lds) ^ (ks << 5)) + kb * 32 * C::ROWB;
        kf[kb][ks] = *(const V8*)(k_stage + at);
        vf[kb][ks] = *(const V8*)(v_stage + at);
      }
    lds_barrier();  // (every wave has read before a first step's loads overwrite)
  } else {
    __syncthreads();
  }

  // byte of a lane's 16 in a 1 KiB piece of a dS unit: [key l32][query group g]
  const int ds_lane = l32 * 32 + g * 16;
  // dS of a step, packed to 16 bits as the operand of its dK MFMAs.  HAND: the four groups also
  // go to the step's dS unit -- under the first MFMAs of the NEXT step (stores issued late in
  // their own step would still be on their way at its end, and the wait for the tile loads
  // there waits for every vector memory operation of the wave: that cost a fifth of the
  // kernel).  ds_pend = where they go: the unit of the last computed step, or nowhere.
  // (WALK4 has no registers for the carry and stores in the same step.)
  constexpr bool CARRY = HAND && !WALK4;
  [[maybe_unused]] V8 ds_carry[KB][2];
  [[maybe_unused]] int ds_pend = kDsNowhere;
  auto store_ds = [&](const V8(&from)[KB][2], int pc, int voff) __attribute__((always_inline)) {
    // piece [key block][query half] of the unit, 1 KiB per wave instruction: a key's 32 bytes
    // side by side ([query group g][rows 16 ks2 + 4 g .., 16 ks2 + 8 + 4 g ..])
    u32x4 bits;
    __builtin_memcpy(&bits, &from[pc >> 1][pc & 1], 16);
    // (aux 2 = non-temporal: the tiles are read once, by another kernel, much later; measured
    // 6 % faster than plain stores on a 2.4 GB hand-off)
    __builtin_amdgcn_raw_buffer_store_b128(bits, ds_rsrc, voff + pc * 1024, ds_pend, 2);
  };
  // (the lane's offset, opaque to the optimiser: or it keeps the four sums voff + pc * 1024 in
  // registers across the walk instead of using the instruction's immediate offset)
  auto ds_voff = [&]() __attribute__((always_inline)) {
    int v = ds_lane;
    asm volatile("" : "+v"(v));
    return v;
  };
  // For which first rows i0 of a 32-row tile does any (query, key of this wave) pair survive
  // the mask (need_*), and for which is no pair masked (full_*)?  With
  // i1 = min(i0 + 32, len_q) - 1 and the wave's keys jw0 .. jw1 the conditions
  //   needed: i0 < len_q, jw0 < len_k, jw0 <= i1 + shift + wr, jw1 >= i0 + shift - wl
  //   full:   i0 + 31 < len_q, jw1 < len_k, jw1 <= i0 + shift + wr, jw0 >= i0 + 31 + shift - wl
  // are intervals of i0 whose ends depend on the wave only: a step tests two of them.
  constexpr int kInf = 1 << 30;
  const int need_lo = (a.wr < 0) ? -kInf : jw0 - shift - a.wr - 31;
  int need_hi = min(len_q - 1, (a.wl < 0) ? kInf : jw1 - shift + a.wl);
  if (jw0 >= len_k || (a.wr >= 0 && len_q - 1 < jw0 - shift - a.wr)) need_hi = -kInf - 1;
  const int full_lo = (a.wr < 0) ? -kInf : jw1 - shift - a.wr;
  int full_hi = min(len_q - 32, (a.wl < 0) ? kInf : jw0 - 31 - shift + a.wl);
  if (jw1 >= len_k) full_hi = -kInf - 1;
  const unsigned need_n = (unsigned)max(need_hi - need_lo + 1, 0), full_n = (unsigned)max(full_hi - full_lo + 1, 0);

  // one query tile: prefetch the next one into (qn, don, stn), compute on (qc, doc, stc)
  auto step = [&](int it, const char* qc, const char* doc, const float* stc, char* qn, char* don,
                  float* stn) __attribute__((always_inline)) {
    const int i0 = cur_i0;
    cur_i0 = nxt.i0;  // the tile fetched now is the next step's
    [[maybe_unused]] const int ds_unit = cur_ds;
    cur_ds = nxt.ds;
    const bool has_next = it + 1 < n_iter;
    const float* lse_lds = stc;
    const float* delta_lds = stc + C::BM;
    // (opaque: the XOR forms of the lane offsets are made where they are used, not kept)
    if constexpr (WALK4) asm volatile("" : "+v"(dma_chunk));
    const bool needed = WALK4 || (HAND ? i0 >= need_lo && i0 <= need_hi : (unsigned)(i0 - need_lo) < need_n);
    if (!needed && has_next) {
      static_for<NPART>([&](auto pc) __attribute__((always_inline)) { load_part(pc, qn, don, stn); });
      if (FREE_RUN || it + 2 < n_iter) advance();
    }
    if constexpr (CARRY) {
      if (!needed) {
        const int voff = ds_voff();
#pragma unroll
        for (int pc = 0; pc < 2 * KB; pc++) store_ds(ds_carry, pc, voff);
        ds_pend = kDsNowhere;
      }
    }
    if (needed) {
      const bool full = HAND ? i0 >= full_lo && i0 <= full_hi : (unsigned)(i0 - full_lo) < full_n;
      // The four GEMMs of the (32 queries x 64 keys) sub-tile -- S = Q K^T, dP = dO V^T,
      // dV^T += dO^T P, dK^T += Q^T dS; KB KS MFMAs each, rows = queries, lane = key column
      // -- their LDS reads and the vector work are written out in issue order, one group
      // per MFMA, with scheduling fences between the groups.  Every fragment read from LDS
      // feeds the MFMAs of both key blocks; K and V come from registers; fragments are fetched
      // AH fragment slots ahead; P = exp2(S c - lse2) is computed under the dP MFMAs and
      // dS = P (dP - delta) under the dV MFMAs; dP - delta comes out of the MFMAs, whose
      // chains start from -delta in the accumulator layout.
      constexpr int NG = KB * KS;   // MFMAs per GEMM (KS = 2 DB)
      constexpr int NF = 4 * KS;    // fragment slots: Q, dO, dO^T, Q^T; KB MFMAs each
      constexpr int AH = 2;
      constexpr int GPC = NG / (4 * KB);  // MFMA groups per chunk of vector work
      static_assert(KS == 2 * DB && KB == 2, "GEMM shapes");
      auto fence = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
      V8 fa[NF];
      auto fetch = [&](auto fc) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value;
        if constexpr (f < 2 * KS) {
          constexpr int ks = f % KS;
          int at = a_row;
          if constexpr (WALK4 && ks >= KS / 2) asm volatile("" : "+v"(at));
          fa[f] = *(const V8*)((f < KS ? qc : doc) + (at ^ (ks << 5)));
        } else if constexpr (f < NF) {
          constexpr int j = (f - 2 * KS) % KS, ks2 = j / DB, d = j % DB;
          const char* src = f < 3 * KS ? doc : qc;
          const int off0 = (t_row0 ^ (d << 6)) + ks2 * 16 * C::ROWB;
          const int off1 = (t_row1 ^ (d << 6)) + ks2 * 16 * C::ROWB;
          fa[f] = tr_pair<V8>(src + off0, src + off1);
        }
      };
      f32x16 sacc[KB], pacc[KB];
      // -delta of the 32 rows in the accumulator layout, from which the dP chains start, is read
      // into the second key block's accumulator: the first block's chain takes it as a separate
      // start operand, the second block's chain then accumulates in place
      f32x4 l4[4];   // -lse2 of the rows
      V8 pb[KB][2], ds_step[KB][2];
      V8(&dsb)[KB][2] = *[&]() __attribute__((always_inline)) {
        if constexpr (CARRY) return &ds_carry;  // lives on into the next step
        else return &ds_step;
      }();
      // vector work in 2 KB chunks of four rows: chunk order lets the packed operands of
      // the first k-step be complete first
      auto chunk_of = [](int c, int& kb, int& i4) __attribute__((always_inline)) {
        kb = (c >> 1) & 1;
        i4 = (c & 1) | ((c >> 2) << 1);
      };
      // P stays in vector registers from here to dS (the S / dP accumulators live in
      // accumulation registers, which the vector ALU reaches only through copies)
      float pk[KB][16];
      auto p_chunk = [&](auto cc) __attribute__((always_inline)) {
        int kb, i4;
        chunk_of(decltype(cc)::value, kb, i4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int i = 4 * i4 + e;
          pk[kb][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][i], a.scale_log2, l4[i4][e]));
        }
        if (i4 & 1) pb[kb][i4 >> 1] = M::pack(&pk[kb][8 * (i4 >> 1)]);
      };
      float dsk[KB][8];  // dS of the current pair of chunks
      auto ds_chunk = [&](auto cc) __attribute__((always_inline)) {
        int kb, i4;
        chunk_of(decltype(cc)::value, kb, i4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int i = 4 * i4 + e;
          dsk[kb][4 * (i4 & 1) + e] = pk[kb][i] * pacc[kb][i];  // zero where P is
        }
        if (i4 & 1) dsb[kb][i4 >> 1] = M::pack(dsk[kb]);
      };

      [[maybe_unused]] int ds_voff_step = 0;
      if constexpr (CARRY) ds_voff_step = ds_voff();
      static_for<AH>([&](auto fc) __attribute__((always_inline)) { fetch(fc); });
      fence();
      static_for<4 * NG>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = decltype(mc)::value;
        constexpr int f = m / KB, kb = m % KB;  // fragment slot and key block of this MFMA
        if constexpr (kb == 0) fetch(std::integral_constant<int, f + AH>{});
        // (no branch around every load: past the last tile what the cursor is on, that tile or, where it runs
        // on (FREE_RUN), one at the start of the head's walk, is fetched once more into idle buffers)
        // (WALK4 issues four times as many: one every other MFMA)
        constexpr int every = WALK4 ? 2 : 1;
        if constexpr (m % every == 0 && m / every < NPART) load_part(std::integral_constant<int, m / every>{}, qn, don, stn);
        if constexpr (CARRY && m < 2 * KB) {
          store_ds(ds_carry, m, ds_voff_step);
          if constexpr (m == 2 * KB - 1) ds_pend = ds_unit;
        }
        // row statistics: -delta early in S (the dP chains start from it), -lse2 at its end
        if constexpr (m >= 4 && m < 8) {
          const f32x4 t4 = *(const f32x4*)(delta_lds + 8 * (m - 4) + 4 * g);
#pragma unroll
          for (int e = 0; e < 4; e++) pacc[KB - 1][4 * (m - 4) + e] = t4[e];
        }
        if constexpr (m >= NG - 4 && m < NG) l4[m - (NG - 4)] = *(const f32x4*)(lse_lds + 8 * (m - (NG - 4)) + 4 * g);
        if constexpr (m < NG) {
          if constexpr (f == 0) {
            if (full) {
              M::mfma32_vec0(fa[f], kf[kb][f], sacc[kb]);
            } else {
              // The mask enters as the start value of the S chain: 0 for a visible pair, -inf
              // otherwise (P = exp2(-inf) = 0, hence dS = 0).  Row r = c + 4 g of the tile, c
              // fixed per register, is visible from key jc iff rmin <= r <= rmax with
              //   rmin = t - rel_hi, rmax = min(t - rel_lo, rows_ok - 1), t = jc - i0 - shift:
              // one unsigned comparison of r - rmin against the width of that interval.
              constexpr int kBig = 1 << 29;  // |t| stays below it
              const int rel_lo = (a.wl < 0) ? -kBig : -a.wl;
              const int rel_up = (a.wr < 0) ? kBig : a.wr;
              int lane_m = lane;
              if constexpr (WALK4) {  // (taken afresh in this rare path: no register for it)
                lane_m = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
                asm volatile("" : "+v"(lane_m));
              }
              const int jc = jw0 + kb * 32 + (lane_m & 31);
              const int t = jc - i0 - shift;
              const int rows_ok = (jc < len_k) ? len_q - i0 : 0;  // rows r < rows_ok are real
              const int rmin = t - rel_up;
              const int rmax = min(t - rel_lo, rows_ok - 1);
              const unsigned width = (unsigned)max(rmax - rmin + 1, 0);
              const int base = 4 * (lane_m >> 5) - rmin;
              select_lanes<16>(
                  [&](auto nc) __attribute__((always_inline)) {
                    constexpr int i = decltype(nc)::value;
                    return lanes((unsigned)(base + 8 * (i >> 2) + (i & 3)) < width);
                  },
                  [&](auto nc, bool v) __attribute__((always_inline)) {
                    sacc[kb][decltype(nc)::value] = v ? 0.f : -__builtin_inff();
                  });
              M::mfma32_vec(fa[f], kf[kb][f], sacc[kb]);
            }
          } else {
            M::mfma32_vec(fa[f], kf[kb][f], sacc[kb]);
          }
        } else if constexpr (m < 2 * NG) {
          if constexpr (f == KS) {
            if constexpr (kb < KB - 1) {
              M::mfma32_vec_init(fa[f], vf[kb][f - KS], pacc[KB - 1], pacc[kb]);
            } else {
              M::mfma32_vec(fa[f], vf[kb][f - KS], pacc[kb]);
            }
          } else {
            M::mfma32_vec(fa[f], vf[kb][f - KS], pacc[kb]);
          }
          if constexpr ((m - NG + 1) % GPC == 0) p_chunk(std::integral_constant<int, (m - NG + 1) / GPC - 1>{});
        } else if constexpr (m < 3 * NG) {
          constexpr int j = f - 2 * KS, ks2 = j / DB, d = j % DB;
          dv_acc[kb][d] = M::mfma32(fa[f], pb[kb][ks2], dv_acc[kb][d]);
          if constexpr ((m - 2 * NG + 1) % GPC == 0)
            ds_chunk(std::integral_constant<int, (m - 2 * NG + 1) / GPC - 1>{});
        } else {
          constexpr int j = f - 3 * KS, ks2 = j / DB, d = j % DB;
          dk_acc[kb][d] = M::mfma32(fa[f], dsb[kb][ks2], dk_acc[kb][d]);
          if constexpr (HAND && WALK4 && m < 3 * NG + 2 * KB) {
            if constexpr (m == 3 * NG) {
              ds_pend = ds_unit;
              ds_voff_step = ds_voff();
            }
            store_ds(dsb, m - 3 * NG, ds_voff_step);
          }
        }
        fence();
      });
      if (FREE_RUN || it + 2 < n_iter) advance();
    }
    if constexpr (WALK4) wait_vmem_but<0>();  // the wave's own tiles: nobody else reads them
    else __syncthreads();
  };

  for (int it = 0; it < n_iter; it += 2) {
    step(it, qb0, dob0, stb0, qb1, dob1, stb1);
    if (it + 1 < n_iter) step(it + 1, qb1, dob1, stb1, qb0, dob0, stb0);
  }
  if constexpr (CARRY) {  // the last computed step's dS
    const int voff = ds_voff();
#pragma unroll
    for (int pc = 0; pc < 2 * KB; pc++) store_ds(ds_carry, pc, voff);
  }

  // ---- write dK, dV (C layout: lane = key, regs = d) -----------------------------------
  // The lane's position is taken afresh (opaque to the optimiser): addresses derived from
  // values computed before the walk would be kept in registers across it, and spilled.
  int lane_e = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  asm volatile("" : "+v"(lane_e));
  const int l32_e = lane_e & 31, g_e = lane_e >> 5;
  if constexpr (WALK4) {
    // The four waves' sums of the block's 64 keys meet in LDS as fp32, one matrix at a time: a
    // wave's 64 x D values fill its own tile buffers (row = key, chunk c of 16 bytes at position
    // c ^ (key mod chunks-per-row)); then all threads add the four parts in wave order, 8 values
    // each, and store whole rows.
    static_assert(W_LDS == 64 * D * 4, "a matrix of 64 keys in fp32 fills a wave's tile buffers");
    constexpr int FPR = D / 4;  // fp32 chunks per row
#pragma unroll
    for (int mtx = 0; mtx < 2; mtx++) {
      const float sc = mtx == 0 ? a.scale : 1.f;
#pragma unroll
      for (int kb = 0; kb < KB; kb++)
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
          for (int i4 = 0; i4 < 4; i4++) {
            const f32x16& acc = mtx == 0 ? dk_acc[kb][d] : dv_acc[kb][d];
            const f32x4 val = {acc[4 * i4], acc[4 * i4 + 1], acc[4 * i4 + 2], acc[4 * i4 + 3]};
            const int c = d * 8 + 2 * i4 + g_e;
            *(f32x4*)(q_s0 + wave * W_LDS + (kb * 32 + l32_e) * (D * 4) + ((c ^ (l32_e & (FPR - 1))) << 4)) = val;
          }
      __syncthreads();
      void* const dst = mtx == 0 ? dk_buf : dv_buf;
      const int64_t dst_off = mtx == 0 ? dk_off : dv_off;
      const int64_t dst_st = mtx == 0 ? a.dk_st[1] : a.dv_st[1];
      constexpr int RPI = 256 / C::CPR;
      const int row0 = (wave * 64 + lane_e) / C::CPR, c = (lane_e % C::CPR) * 2;
      put_rows<T, RPI, 64 / RPI>(
          dst, dst_off + (int64_t)(j0 + row0) * dst_st + c * 4, dst_st, len_k - j0 - row0, j0 + 63 < len_k, a.wide_dkv,
          a.dkv_accumulate, [&](int n) {
            const int row = row0 + n * RPI;
            const char* src = q_s0 + row * (D * 4);
            const int at0 = (c ^ (row & (FPR - 1))) << 4, at1 = ((c + 1) ^ (row & (FPR - 1))) << 4;
            f32x4 lo = *(const f32x4*)(src + at0), hi = *(const f32x4*)(src + at1);
#pragma unroll
            for (int w = 1; w < 4; w++) {
              lo += *(const f32x4*)(src + w * W_LDS + at0);
              hi += *(const f32x4*)(src + w * W_LDS + at1);
            }
            const float x[8] = {lo[0] * sc, lo[1] * sc, lo[2] * sc, lo[3] * sc,
                                hi[0] * sc, hi[1] * sc, hi[2] * sc, hi[3] * sc};
            return M::pack(x);
          });
      __syncthreads();
    }
    return;
  }
  // Through LDS, one 32-key block of one matrix at a time: in the accumulator layout a lane
  // holds 4 consecutive d of one key, so a direct store instruction would touch 32 rows with
  // 16 bytes each (256 such instructions per block; at short walks -- 40 steps per block at
  // window 1000 and one q head per kv head -- they took a tenth of the kernel).  Each wave
  // stages its block in the tile buffer nobody reads any more (rows of 16-byte chunks, chunk
  // c of row r at position c ^ (r % chunks-per-row)), and stores whole rows, 16 bytes a lane.
  char* stage = wave == 0 ? q_s0 : wave == 1 ? q_s1 : wave == 2 ? do_s0 : do_s1;
  static_assert(C::Q_TILE >= 32 * C::ROWB, "a 32-key block fits a tile buffer");
  const int wr_row = l32_e * C::ROWB + g_e * 8;
  const int wr_swz = l32_e & (C::CPR - 1);
#pragma unroll
  for (int mtx = 0; mtx < 2; mtx++)
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      const float sc = mtx == 0 ? a.scale : 1.f;
#pragma unroll
      for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i4 = 0; i4 < 4; i4++) {
          const f32x16& acc = mtx == 0 ? dk_acc[kb][d] : dv_acc[kb][d];
          *(typename M::V4*)(stage + wr_row + (((d * 4 + i4) ^ wr_swz) << 4)) =
              M::pack4(acc[4 * i4] * sc, acc[4 * i4 + 1] * sc, acc[4 * i4 + 2] * sc,
                       acc[4 * i4 + 3] * sc);
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own writes have landed
      void* const dst = mtx == 0 ? dk_buf : dv_buf;
      const int64_t dst_off = mtx == 0 ? dk_off : dv_off;
      const int64_t dst_st = mtx == 0 ? a.dk_st[1] : a.dv_st[1];
      constexpr int RPI = 64 / C::CPR;
      const int row0 = lane_e / C::CPR, c = lane_e % C::CPR;
      const int64_t at = dst_off + (int64_t)(jw0 + kb * 32 + row0) * dst_st + c * 8;
      put_rows<T, RPI, 32 / RPI>(dst, at, dst_st, len_k - jw0 - kb * 32 - row0, jw0 + kb * 32 + 31 < len_k,
                                 a.wide_dkv, a.dkv_accumulate, [&](int n) {
                                   const int row = row0 + n * RPI;
                                   return *(const V8*)(stage + row * C::ROWB + ((c ^ (row & (C::CPR - 1))) << 4));
                                 });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next block overwrites
    }
}

// ============================================================================
// dK / dV of sink keys
// ============================================================================
// With sink keys and a bounded window, key j < n_sink is seen by every later row of its
// sequence: a few keys against all the rows, far too thin for the dK/dV kernel's tiles.  Left to that
// kernel, the first key tile of every sequence walked every query tile with one wave of four
// at work and took several times as long as any other block (a pack of 65536 tokens in four
// sequences: 10.8 ms, a third of it that tail).  So the dK/dV kernel treats sink keys like any
// other key (band pairs only), and this kernel, which runs after it, computes the sink keys'
// complete dK / dV -- all the rows that see them, inside the window and beyond -- and overwrites those
// few rows of dk / dv:
//   s = q . k_j, P = exp2(s c - lse2), dP = dO . v_j, dS = P (dP - delta)
//   dV_j = sum P dO, dK_j = scale sum dS q
// A wave takes 16 rows of one q head at a time, fetched one tile ahead: Q and dO as B operands (lane =
// row l % 16, 8 consecutive d at 32 ks + 8 (l / 16)), four sinks repeated four times as the A operand, so
// that after KS MFMAs each lane holds s and dP - delta of its own row for all four of them, and
// multiplies them in fp32 into its own 2 x D / 4 sums per sink.  (P and dS stay fp32: as MFMA operands they
// would be 16 bits.)  256 registers hold the sums of two sinks: with more than one, pairs of waves share the
// rows and take two sinks each.  The sums of a block, over the 16 rows of a tile and its waves,
// leave through LDS in a fixed order.
// A unit (sequence, kv head) of up to sink_chunks chunks of tiles; with more than one, their sums go to the
// workspace as fp32 [unit][chunk][sink][dK, dV][D], and the block of a unit that arrives
// last adds the chunks in chunk order and writes the rows (the same order whichever block that is, so
// the result does not depend on timing, and nobody waits).
// Bound by reading Q and dO once where there are many rows, by latencies where there are few.
// The earlier form, whose lanes held 8 d of a row and summed every dot product across 16 lanes, walked 512
// rows of each head of the group in one block without fetching ahead.  us, before / now (traced), this launch
// and the dK/dV launch ahead of it: 2 x 300 rows, 32 / 8 heads, window 100, 1 sink 75 / 29; 12053 rows, 8 / 2
// heads, window 67, 1 sink 142 / 57; 2 x 31793 rows, 16 / 4 heads, window 1000, 4 sinks 1168 / 1102; 550
// sequences of 20 tokens, 12 heads, 1 sink 565 / 269; this launch alone: 65536 tokens in four sequences, 32 / 8
// heads, 4 sinks 389 / 304 (3.6 TB/s); packs of one long sequence among 63 of 16 tokens, 4 sinks, window 256:
// 32000 tokens, 32 = 32 heads (2048 units of one chunk, so that 32 blocks have the long sequence) 1086 / 920,
// 16000 tokens, 8 / 2 heads 2924 / 206.

// sum over the aligned group of 16 lanes, in every lane of the group
__device__ __forceinline__ float lane_group_sum16(float x) {
  auto dpp = [](float v, auto ctrl) __attribute__((always_inline)) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), decltype(ctrl)::value,
                                                       0xf, 0xf, true));
  };
  x += dpp(x, std::integral_constant<int, 0x140>{});  // row_mirror
  x += dpp(x, std::integral_constant<int, 0x141>{});  // row_half_mirror
  x += dpp(x, std::integral_constant<int, 0x1b>{});   // quad_perm 3 2 1 0
  x += dpp(x, std::integral_constant<int, 0xb1>{});   // quad_perm 1 0 3 2
  return x;
}

// NS: sinks of a wave, 1 (the waves of a block share out the tiles) or 2 (pairs of waves do, and the
// waves of a pair take sinks 0, 1 and 2, 3 of every four)
template <typename T, int D, int NS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void attn_bwd_sink_kernel(const AttnArgs a) {
  using M = Mma<T>;
  using V8 = typename M::V8;
  constexpr int KS = D / 32;
  constexpr int SG = NS;        // groups of sinks in the block (waves of a pair)
  constexpr int RW = 4 / SG;    // waves that share out the tiles
  constexpr int NB = NS * SG;   // sinks of a pass
  __shared__ float red_s[4][NS * 2 * D];
  __shared__ __attribute__((aligned(16))) T k_s[SG * 4 * D], v_s[SG * 4 * D];  // the pass's sinks, NS of every four rows

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, u = lane >> 4;
  const int sg = wave & (SG - 1), rw = wave / SG;
  const int c = blockIdx.x % a.sink_chunks;
  const int unit = blockIdx.x / a.sink_chunks;  // (sequence, kv head)
  const int hk = unit % a.heads_kv, b = unit / a.heads_kv;
  int64_t q_row0 = 0, k_row0 = 0;
  int len_q = a.seqlen_q, len_k = a.seqlen_k;
  if (a.cu_q) {
    q_row0 = a.cu_q[b];
    k_row0 = a.cu_k[b];
    len_q = a.cu_q[b + 1] - a.cu_q[b];
    len_k = a.cu_k[b + 1] - a.cu_k[b];
  }
  const int ns_all = min(a.n_sink, len_k);
  // the unit's tiles in n_chunks chunks (at most a.sink_chunks, of two tiles per wave or
  // more)
  const int n_rt = (len_q + 15) >> 4, total = n_rt * a.group;
  const int per = max((total + a.sink_chunks - 1) / a.sink_chunks, 2 * RW);
  const int n_chunks = (total + per - 1) / per;
  if (c >= n_chunks || ns_all == 0) return;
  const int shift = a.shift_explicit ? a.shift_val : len_k - len_q;
  const int t_end = min(total, (c + 1) * per);

  const T* q_ptr = (const T*)a.q + b * a.q_st[0] + q_row0 * a.q_st[1] + hk * a.group * a.q_st[2] + u * 8;
  const T* do_ptr = (const T*)a.dout + b * a.do_st[0] + q_row0 * a.do_st[1] + hk * a.group * a.do_st[2] + u * 8;
  const T* k_ptr = (const T*)a.k + b * a.k_st[0] + k_row0 * a.k_st[1] + hk * a.k_st[2];
  const T* v_ptr = (const T*)a.v + b * a.v_st[0] + k_row0 * a.v_st[1] + hk * a.v_st[2];
  const int64_t ws_row0 = (int64_t)hk * a.group * a.rows_q + (a.cu_q ? q_row0 : (int64_t)b * a.seqlen_q);
  T* dk_ptr = (T*)a.dk + b * a.dk_st[0] + k_row0 * a.dk_st[1] + hk * a.dk_st[2];
  T* dv_ptr = (T*)a.dv + b * a.dv_st[0] + k_row0 * a.dv_st[1] + hk * a.dv_st[2];
  auto put = [&](int j, int at, float sum) __attribute__((always_inline)) {  // at: d of dK, then of dV
    if (at < D) dk_ptr[(int64_t)j * a.dk_st[1] + at] = (T)(sum * a.scale);
    else dv_ptr[(int64_t)j * a.dv_st[1] + at - D] = (T)sum;
  };

  auto publish = [](float* at, float x) __attribute__((always_inline)) {
    __hip_atomic_store(at, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  struct Tile {
    V8 q[KS], d[KS];
    float nl, nd;  // the row's statistics, stored negated
    int row;
  };
  for (int j0 = 0; j0 < ns_all; j0 += NB) {
    const int jb = j0 + sg * NS;  // the wave's sinks: jb .. jb + NS - 1
    if (j0 > 0) __syncthreads();  // the previous pass's readers are done
    for (int idx = tid; idx < SG * 4 * D; idx += 256) {
      const int row = idx / D, j = j0 + (row >> 2) * NS + (row & 3);
      const bool real = (row & 3) < NS && j < ns_all;
      k_s[idx] = real ? k_ptr[(int64_t)j * a.k_st[1] + idx % D] : (T)0.f;
      v_s[idx] = real ? v_ptr[(int64_t)j * a.v_st[1] + idx % D] : (T)0.f;
    }
    float acck[NS][KS * 8], accv[NS][KS * 8];
#pragma unroll
    for (int i = 0; i < NS; i++)
#pragma unroll
      for (int e = 0; e < KS * 8; e++) acck[i][e] = accv[i][e] = 0.f;
    int t = c * per + rw;
    __syncthreads();
    if (jb < ns_all && t < t_end) {
      // cursor: tile rt of the unit's q head h, the heads of a tile's rows one after the other, which lie side
      // by side in memory (the loads of a tile behind the chunk's last are those of the last, and not used)
      int rt = t / a.group, h = t - rt * a.group;
      auto fetch = [&](Tile& x) __attribute__((always_inline)) {
        x.row = rt * 16 + r;
        const int row = min(x.row, len_q - 1);
        const T* q_row = q_ptr + h * a.q_st[2] + (int64_t)row * a.q_st[1];
        const T* do_row = do_ptr + h * a.do_st[2] + (int64_t)row * a.do_st[1];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          x.q[ks] = *(const V8*)(q_row + ks * 32);
          x.d[ks] = *(const V8*)(do_row + ks * 32);
        }
        x.nl = a.lse2[ws_row0 + h * a.rows_q + row];
        x.nd = a.delta[ws_row0 + h * a.rows_q + row];
      };
      Tile cur, nxt;
      fetch(cur);
      for (; t < t_end; t += RW) {
        if (t + RW < t_end) {
          h += RW;
          while (h >= a.group) {
            h -= a.group;
            rt++;
          }
        }
        fetch(nxt);
        // rows past the end, which hold the last row's values: their P and dS are zero, but zero times an
        // infinity or a NaN of that row is a NaN
        if (__builtin_amdgcn_readfirstlane(cur.row - r) + 16 > len_q) {
#pragma unroll
          for (int ks = 0; ks < KS; ks++)
            if (cur.row >= len_q) cur.q[ks] = cur.d[ks] = V8{0, 0, 0, 0, 0, 0, 0, 0};
        }
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = {cur.nd, cur.nd, cur.nd, cur.nd};
        int a_row = (sg * 4 + (r & 3)) * D + u * 8;  // row r of the A operand: sink r % 4
        asm volatile("" : "+v"(a_row));              // (read here: kept in registers the operands would spill)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          s = M::mfma16(*(const V8*)(k_s + a_row + ks * 32), cur.q[ks], s);
          dp = M::mfma16(*(const V8*)(v_s + a_row + ks * 32), cur.d[ks], dp);
        }
        const int hi = (a.wr >= 0) ? min(len_k - 1, cur.row + shift + a.wr) : len_k - 1;
        float p[NS], ds[NS];
#pragma unroll
        for (int i = 0; i < NS; i++) {
          const int j = jb + i;
          const bool vis = cur.row < len_q && j < ns_all && j <= hi;  // a sink key: no lower bound
          p[i] = vis ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale_log2, cur.nl)) : 0.f;
          ds[i] = vis ? p[i] * dp[i] : 0.f;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const float qe = (float)cur.q[ks][e], de = (float)cur.d[ks][e];
#pragma unroll
            for (int i = 0; i < NS; i++) {
              acck[i][ks * 8 + e] = __builtin_fmaf(ds[i], qe, acck[i][ks * 8 + e]);
              accv[i][ks * 8 + e] = __builtin_fmaf(p[i], de, accv[i][ks * 8 + e]);
            }
          }
        cur = nxt;
      }
    }
    // the wave's sums over its 16 rows, then the block's over its waves, in wave order
#pragma unroll
    for (int i = 0; i < NS; i++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float k_sum = lane_group_sum16(acck[i][ks * 8 + e]), v_sum = lane_group_sum16(accv[i][ks * 8 + e]);
          if (r == 0) {
            red_s[wave][(i * 2 + 0) * D + ks * 32 + u * 8 + e] = k_sum;
            red_s[wave][(i * 2 + 1) * D + ks * 32 + u * 8 + e] = v_sum;
          }
        }
    __syncthreads();
    for (int idx = tid; idx < NB * 2 * D; idx += 256) {
      const int jj = idx / (2 * D), at = idx % (2 * D);
      if (j0 + jj >= ns_all) break;
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < RW; w++) sum += red_s[w * SG + jj / NS][(jj % NS) * 2 * D + at];
      if (n_chunks == 1) put(j0 + jj, at, sum);
      else publish(a.sink_part + ((int64_t)unit * a.sink_chunks + c) * (a.n_sink * 2 * D) + (j0 + jj) * (2 * D) + at, sum);
    }
  }
  if (n_chunks == 1) return;
  // Count this chunk in; the last one of the unit adds them all up.  The sums are written through to where
  // every XCD reads them and read from there, each by itself: a fence would write back and then drop
  // the XCD's whole L2, under the feet of the blocks that are at work, for every block.  That rests on the
  // hardware, not on the language, in which relaxed operations order nothing: on gfx950 a store of device
  // scope is written through, s_waitcnt vmcnt(0) waits until it has arrived there, and the barrier
  // puts every wave's wait ahead of the count (us, this launch,
  // with a fence per block / so: 51330 tokens in long sequences, 32 / 8 heads, head_dim 64, 191 / 105; 65536
  // tokens, 4 sinks, 390 / 316; 3 x 5000 rows, 32 heads, head_dim 64, 105 / 60; with four times the blocks the
  // fences cost 382 and 670).
  __shared__ int arrived_s;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) arrived_s = __hip_atomic_fetch_add(a.sink_count + unit, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (arrived_s != n_chunks - 1) return;
  if (tid == 0) a.sink_count[unit] = 0;  // the next launch on this workspace starts from zero
  const float* parts = a.sink_part + (int64_t)unit * a.sink_chunks * (a.n_sink * 2 * D);
  for (int idx = tid; idx < ns_all * 2 * D; idx += 256) {
    float sum = 0.f;
#pragma unroll 8
    for (int cc = 0; cc < n_chunks; cc++)
      sum += __hip_atomic_load(parts + (int64_t)cc * (a.n_sink * 2 * D) + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    put(idx / (2 * D), idx % (2 * D), sum);
  }
}

// ============================================================================
// dQ
// ============================================================================
// LDS read-ahead of the dQ kernel's two matrix sections, in fragments (measured: 7 / 4 and
// 6 / 4 are equal, 12 / 6 is 2-3 % slower; 8 / 4 spills at head_dim 128 -- all 256 registers of
// a lane are in use in the first section once S^T and dP^T are both live -- and is 5 % slower)
#ifndef RSWA_DQ_AH1
#define RSWA_DQ_AH1 7
#endif
#ifndef RSWA_DQ_AH2
#define RSWA_DQ_AH2 4
#endif
// dQ launches of head_dim 128 whose rows see at most this many keys on average, and all of head_dim 64, use
// blocks of 4 waves, two per compute unit (three at head_dim 64, against which a block of 8 is slower at any
// length: us, 8 / 4 waves, 32768 rows, 32 / 8 heads, window 4096, 1546 / 1301; 12000 rows, 28 / 4 heads, causal
// without a window, 1082 / 834; 20000 rows, 8 heads, window 4096, 272 / 219; head_dim 128, 32 / 8 heads:
// window 256 -22 %, window 1000 -8 %, the rank step with its half-empty previous-chunk block -1.4 %;
// sequences of 16384 and more rows at window 4096 +1 %; 32 = 32 heads, window 1000: -2 %)
#ifndef RSWA_DQ_SMALL_AVG_KEYS
#define RSWA_DQ_SMALL_AVG_KEYS 3200
#endif
template <int D>
struct DqCfg {
  static constexpr int BN = 64;  // keys per step
  static constexpr int KS = D / 32;   // k-steps of the 16x16x32 MFMAs over the head dim
  static constexpr int DB = D / 16;   // 16-row blocks of dQ^T
  static constexpr int KBLK = BN / 16;  // 16-key blocks per tile
  static constexpr int CPR = D / 8;
  static constexpr int ROWB = D * 2;
  static constexpr int TILE = BN * ROWB;
  static constexpr int O_STRIDE = D * 2 + 16;
  static_assert(TILE >= 32 * O_STRIDE, "one wave's epilogue staging fits one tile buffer");
};

// Waves per SIMD that the dQ kernel is built for.  At head_dim 64 blocks of 4 waves fit three times into
// a compute unit, with 164 registers and a shorter read-ahead (3 / 2; 7 / 4 would spill): half the MFMAs
// per score leave the vector work and its latencies as the bound, which a third wave fills (us, dQ with
// statistics, two / three: 2 x 31654 rows, 28 / 4 heads, window 100, 308 / 245; 2 x 7078, window 570, 120 /
// 104; 15510 rows, 16 / 4 heads, window 990, 112 / 106; launches that two blocks per unit hold +-1 %).
template <int D, int NW>
constexpr int dq_waves = D == 64 && NW == 4 ? 3 : 2;

// The key tile table of a pack, by one block: running sums of the sequences' tile counts, THREADS
// sequences at a time (a scan in each wave, the waves' totals through LDS).
template <int THREADS>
__device__ __forceinline__ void write_ktile(const AttnArgs& a, int* wave_sum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int first_n = (a.cu_k[1] - a.cu_k[0] + (1 << a.ktile_log2) - 1) >> a.ktile_log2;
  int period = 0;  // tiles (of this thread's sequences) for which the snake order is
  int base = 0;
  for (int b0 = 0; b0 < a.batch; b0 += THREADS) {
    const int b = b0 + (int)threadIdx.x;
    const int len = b < a.batch ? a.cu_k[b + 1] - a.cu_k[b] : 0;
    const int n = (len + (1 << a.ktile_log2) - 1) >> a.ktile_log2;
    int sum = n;  // inclusive
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int up = __shfl_up(sum, m, 64);
      if (lane >= m) sum += up;
    }
    __syncthreads();  // (wave_sum of the previous pass has been read)
    if (lane == 63) wave_sum[wave] = sum;
    __syncthreads();
    int before = base;
    for (int w = 0; w < THREADS / 64; w++) {
      if (w < wave) before += wave_sum[w];
      base += wave_sum[w];
    }
    if (b < a.batch) a.ktile[b] = before + sum - n;
    const bool in_step = a.ktile_log2 == 8 ? (n & 3) == 0 : n == first_n;
    if (in_step && n << a.ktile_log2 <= kSnakeKeys) period += n;
  }
  __syncthreads();
  if (threadIdx.x == 0) wave_sum[0] = 0;
  __syncthreads();
  if (period) atomicAdd(wave_sum, period);
  __syncthreads();
  if (threadIdx.x == 0) {
    a.ktile[a.batch] = base;
    // (28 sequences of 900 to 1083 tokens, 0.77 of the 256-key tiles in fours: 625 us plain, 538 snake;
    // drawn packs of which less than that are: 0.8 % slower by it on average, up to 32 %)
    a.ktile[a.batch + 1] = base > 0 && (int64_t)wave_sum[0] * 10 >= (int64_t)base * 7;
  }
}

// The table alone, for a dK/dV launch whose statistics came with another call: that call's table may
// be of another tile size or lie elsewhere, and the kernel takes its block count and rows from it.
__global__ __launch_bounds__(256) void attn_bwd_ktile_kernel(const AttnArgs a) {
  __shared__ int wave_sum[4];
  write_ktile<256>(a, wave_sum);
}

// What the statistics kernel leaves in the workspace of a pack or a call with sink keys beside the
// statistics of the rows, by one block: the sink kernel's arrival counters at zero, the neutral
// value behind a pack's lse2 array, the neutral pair for the rows after a pack's last that the
// tile kernels read with its last tile, and the key tile table.  (Inside the dQ kernel it would push that kernel's registers into scratch memory.)
__global__ __launch_bounds__(256) void attn_bwd_rest_kernel(const AttnArgs a) {
  __shared__ int wave_sum[4];
  for (int i = threadIdx.x; i < a.n_count; i += 256) a.sink_count[i] = 0;
  if (a.cu_q) {
    const int64_t used = a.rows_q * a.heads_q;
    if (used + threadIdx.x < a.delta - a.lse2) a.lse2[used + threadIdx.x] = -__builtin_inff();
    const int64_t owned = a.cu_q[a.batch];
    const int n = (int)min((int64_t)kStatTileRows, a.rows_q - owned);
    for (int i = threadIdx.x; i < n * a.heads_q; i += 256) {
      const int64_t at = (int64_t)(i / n) * a.rows_q + owned + i % n;
      a.lse2[at] = -__builtin_inff();
      a.delta[at] = -0.f;
    }
  }
  if (a.ktile) write_ktile<256>(a, wave_sum);
}

// Built on v_mfma_f32_16x16x32 (with random operands the matrix pipes sustain about 14 % more
// of these than of the 32x32x16 form before the power limit pulls the clock down).  A wave
// owns 32 query rows as two 16-column blocks: lane l holds query column l % 16 of each block;
// its 8-element fragments cover d = 32 ks + 8 (l / 16) ...; a 64-key tile is four 16-key
// blocks, and S^T / dP^T tiles hold keys 16 kb + 4 (l / 16) + i in element i.  Two such tiles
// of neighbouring key blocks, packed, are the B operand of dQ^T += K^T dS^T over a 32-key slab
// (k order: four keys of the first block, then four of the second); the A operand follows the
// same order: two transposing reads, one per key block.
//
// NW = 8: one block of 8 waves per compute unit (two waves per SIMD).  NW = 4: blocks of 4 waves, two of
// them per compute unit at head_dim 128, three at 64 (dq_waves) -- a SIMD's waves are from independent
// blocks, so that one block's prologue (kernel arguments, a pack's sequence, then the first tiles and the
// rows' own data at once: two or three round trips to memory) and epilogue run under the others' tiles; the
// price is that a K / V tile serves half as many rows.
//
// STATS: the kernel also makes the row statistics of the backward, which it has to read dO for
// anyway, and writes them for the dK/dV kernel, launched after it.  Same bits as the statistics
// kernel's (same order of sums).  What falls away is the second read of dO and a launch; us, statistics +
// dQ, bf16, head_dim 128, two kernels / one: 2 x 8192 rows, 32 / 32 heads, window 1000 457 / 444; a pack of
// 16384 tokens in sequences of 16 to 1024, 32 / 8 heads, 213 / 206; 4001 rows, window 1024, 105 / 99.
template <typename T, int D, bool FAR, int NW, bool STATS>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(dq_waves<D, NW>, dq_waves<D, NW>)))
void attn_bwd_dq_kernel(const AttnArgs a) {
  using C = DqCfg<D>;
  constexpr bool THREE = dq_waves<D, NW> == 3;
  static_assert(NW == 8 || NW == 4, "waves per block");
  static_assert(!(FAR && STATS), "statistics in the first addressing form only");
  constexpr int HSH = NW == 8 ? 2 : 1;  // waves per q head in pair mode: 1 << HSH
  using M = Mma<T>;
  using V8 = typename M::V8;
  constexpr int KS = C::KS, DB = C::DB, KBLK = C::KBLK;
  __shared__ __attribute__((aligned(1024))) char k_s0[C::TILE];
  __shared__ __attribute__((aligned(1024))) char k_s1[C::TILE];
  __shared__ __attribute__((aligned(1024))) char v_s0[C::TILE];
  __shared__ __attribute__((aligned(1024))) char v_s1[C::TILE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15;   // column (query) / row (key, d) inside a 16 block
  const int u = lane >> 4;   // k group

  // pair mode: waves 0-3 and 4-7 take the same 128 rows of two neighbouring q heads;
  // row mode: the 8 waves take 256 consecutive rows of one q head
  const bool pair = (a.group & 1) == 0;
  const int units = pair ? a.group >> 1 : a.group;
  const int bm = pair ? 16 * NW : 32 * NW;
  int rest, hu;
  if (!tile_of_block(a, units, rest, hu)) return;
  const int tiles_before = quotient(rest, a.by_tile);
  const int tile = rest - tiles_before * a.n_tile;
  const int slot = a.rev_q ? a.n_tile - 1 - tile : tile;
  rest = quotient(tiles_before, a.by_heads);  // batch entry (dense)
  const int hk = tiles_before - rest * a.heads_kv;
  const int hq = hk * a.group + (pair ? 2 * hu + (wave >> HSH) : hu);
  SeqInfo s;
  int qt;
  if (a.cu_q) {
    if (!locate_packed(a, slot, (pair ? 4 : 5) + (NW == 8 ? 3 : 2), false, s, qt)) return;
  } else {
    s.batch_idx = rest;
    s.q_row0 = s.k_row0 = 0;
    s.len_q = a.seqlen_q;
    s.len_k = a.seqlen_k;
    qt = slot;
  }
  const int b = s.batch_idx;
  const int len_q = s.len_q, len_k = s.len_k;
  const int i0 = qt * bm;
  if (i0 >= len_q) return;

  const T* q_ptr = (const T*)a.q + b * a.q_st[0] + s.q_row0 * a.q_st[1] + hq * a.q_st[2];
  const T* do_ptr = (const T*)a.dout + b * a.do_st[0] + s.q_row0 * a.do_st[1] + hq * a.do_st[2];
  const T* k_ptr = (const T*)a.k + b * a.k_st[0] + s.k_row0 * a.k_st[1] + hk * a.k_st[2];
  const T* v_ptr = (const T*)a.v + b * a.v_st[0] + s.k_row0 * a.v_st[1] + hk * a.v_st[2];
  const int64_t dq_off = b * a.dq_st[0] + s.q_row0 * a.dq_st[1] + hq * a.dq_st[2];  // (T or fp32)
  const int64_t ws_row0 = a.cu_q ? s.q_row0 : (int64_t)b * a.seqlen_q;

  // ---- key tiles this block visits (same rule as the forward kernel) -----------
  const int i_last = min(i0 + bm, len_q) - 1;
  const KeyTiles tiles = key_tiles<C::BN>(a, i0, i_last, len_q, len_k);
  const int n_tiles = tiles.n_sink + tiles.n_band;
  KeyWalk walk(a, tiles);

  const int r0 = i0 + (pair ? wave & ((1 << HSH) - 1) : wave) * 32;
  const bool wave_valid = r0 < len_q;
  const bool wave_rows_full = r0 + 31 < len_q;
  const RowBounds wb_first = row_bounds(a, r0, len_q, len_k);
  const RowBounds wb_last = row_bounds(a, min(r0 + 31, len_q - 1), len_q, len_k);
  // Tiles, by their first key, that hold keys of the wave's rows, and that all its rows see whole: an interval
  // of the band and one of the sinks each, so that a tile costs a comparison or two.
  // (With this, resources kept instead of selected per tile and the walk's branch: 45 scalar instructions a tile
  // instead of 75, 60 of which both waves of a SIMD issued ahead of their first MFMA.  us, dQ with statistics: the rank
  // step, window 4096, 677 / 667; 2 x 8192 rows, 32 heads, window 1000, 414 / 411; 22 drawn and listed calls 1.0 % on
  // average, single ones of 100 us by nothing or by 4 %.)
  const int need_lo = wb_first.lo - (C::BN - 1);
  const unsigned need_n = wave_valid ? (unsigned)max(wb_last.hi - need_lo + 1, 0) : 0u;
  const int need_sink = wave_valid ? min(a.n_sink, wb_last.hi + 1) : 0;
  const int full_end = wave_rows_full ? wb_first.hi - (C::BN - 1) + 1 : 0;  // behind the last not cut by the upper bound
  const unsigned full_n = (unsigned)max(full_end - wb_last.lo, 0);
  const int full_sink = min(a.n_sink - (C::BN - 1), full_end);

  TileDma<D, C::BN, NW * 64, true> k_dma, v_dma;
  k_dma.init(a.k_st[1], tid);
  v_dma.init(a.v_st[1], tid);
  // (keys in two row ranges: the second range's tensors, at this batch entry and kv head)
  const T* k2_ptr = a.k2 ? (const T*)a.k2 + b * a.k_st[0] + hk * a.k_st[2] : k_ptr;
  const T* v2_ptr = a.v2 ? (const T*)a.v2 + b * a.v_st[0] + hk * a.v_st[2] : v_ptr;
  const KeyRows<T, C::ROWB, FAR> k_rows(k_ptr, k2_ptr, a.seg, len_k, a.k_st[1]), v_rows(v_ptr, v2_ptr, a.seg, len_k, a.v_st[1]);
  auto load_tile = [&](int tile, char* kd, char* vd) __attribute__((always_inline)) {
    const int row = tile * C::BN;
    if constexpr (FAR || THREE) {  // (THREE: the resources would spill)
      k_dma.load(k_rows.template tile<C::BN>(row), kd);
      v_dma.load(v_rows.template tile<C::BN>(row), vd);
    } else if (__builtin_expect(row < a.seg, 1)) {
      k_dma.load(k_rows.first_range(), row * k_rows.stride_bytes, kd);
      v_dma.load(v_rows.first_range(), row * v_rows.stride_bytes, vd);
    } else {  // (code of its own: the first range's resources stay as they are, in registers)
      asm volatile("");
      k_dma.load(k_rows.template tile<C::BN>(row), kd);
      v_dma.load(v_rows.template tile<C::BN>(row), vd);
      asm volatile("");
    }
  };

  // The first tiles are asked for ahead of the rows' own data, and of that everything before the first
  // use: one 16-row half after the other with its statistics, then the tiles, were three round trips to
  // memory, 8 us of a block's start (of 53 at window 1000, of 18 in a pack of short sequences), now 7.
  // us, before / after: a pack of 16384 tokens in sequences of 16 to 1024 189 / 183; rows 8192 with the
  // statistics, window 4096, 664 / 655; 4001 rows, window 1024, 93.7 / 93.1.
  if (n_tiles > 0) load_tile(walk.tile, k_s0, v_s0);

  // Q / dO fragments (B operands) and the (negated) statistics of the lane's two query rows.  The
  // dP^T accumulator chains start from -delta: the MFMAs then deliver dP - delta, and the vector ALU
  // is left with a multiply-add, an exponential, a product and the 16-bit conversion per score.
  // All loads are issued before the first use.  (Rows past the end read the last row's values:
  // their columns are masked in every tile and never stored.)
  V8 qf[2][KS], dof[2][KS];
  float lse2[2];   // -lse2 of the lane's two queries
  f32x4 delta[2];  // -delta of the same, in all four elements (start value of the dP^T chains)
  [[maybe_unused]] V8 of[2][KS];
#pragma unroll
  for (int qb = 0; qb < 2; qb++) {
    const int iq = r0 + 16 * qb + r, row = min(iq, len_q - 1);
    const T* q_row = q_ptr + (int64_t)row * a.q_st[1] + u * 8;
    const T* do_row = do_ptr + (int64_t)row * a.do_st[1] + u * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) dof[qb][ks] = *(const V8*)(do_row + ks * 32);
    if constexpr (STATS) {
      const T* o_row = (const T*)a.out + b * a.o_st[0] + (s.q_row0 + row) * a.o_st[1] + hq * a.o_st[2] + u * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) of[qb][ks] = *(const V8*)(o_row + ks * 32);
      lse2[qb] = a.lse[b * a.lse_st[0] + hq * a.lse_st[1] + (s.q_row0 + row) * a.lse_st[2]];
    } else {
      lse2[qb] = a.lse2[(int64_t)hq * a.rows_q + ws_row0 + row];
      delta[qb][0] = a.delta[(int64_t)hq * a.rows_q + ws_row0 + row];
    }
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[qb][ks] = *(const V8*)(q_row + ks * 32);
  }
  if constexpr (STATS) {
    // the elements behind the lse2 array (see attn_bwd_prep_kernel), where block 0 surely is at
    // work; for a pack, whose first slot may stand for no tile, attn_bwd_rest_kernel writes them
    const int64_t used = a.rows_q * a.heads_q;
    if (!a.cu_q && blockIdx.x == 0 && used + tid < a.delta - a.lse2) a.lse2[used + tid] = -__builtin_inff();
  }
#pragma unroll
  for (int qb = 0; qb < 2; qb++) {
    const int iq = r0 + 16 * qb + r;
    if constexpr (STATS) {
      // delta = sum over d of dO * O: eight elements a time, then the 16 (8) parts of a row
      // pairwise from the farthest, as in the statistics kernel
      float part[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        part[ks] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
          // (products of 16-bit values are exact; contracted, fp16 becomes v_dot2, which rounds
          // otherwise than the statistics kernel)
#pragma clang fp contract(off)
          part[ks] += (float)of[qb][ks][j] * (float)dof[qb][ks][j];
        }
      }
#pragma unroll
      for (int m = KS / 2; m >= 1; m >>= 1)
#pragma unroll
        for (int ks = 0; ks < m; ks++) part[ks] += part[ks + m];
      float sum = part[0];
      sum += __shfl_xor(sum, 32, 64);
      sum += __shfl_xor(sum, 16, 64);
      lse2[qb] = (lse2[qb] == -__builtin_inff()) ? lse2[qb] : -lse2[qb] * kLog2e;
      delta[qb][0] = -sum;
      if (u == 0 && iq < len_q) {
        a.lse2[(int64_t)hq * a.rows_q + ws_row0 + iq] = lse2[qb];
        a.delta[(int64_t)hq * a.rows_q + ws_row0 + iq] = delta[qb][0];
      }
    }
    const float dl = delta[qb][0];
    delta[qb] = f32x4{dl, dl, dl, dl};
  }

  f32x4 dq_acc[DB][2];
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int qb = 0; qb < 2; qb++) dq_acc[d][qb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- lane-constant LDS offsets (swizzle folded: the varying parts are XOR / immediates) ----
  // row fragments of K / V (16-byte reads): row 16 kb + r, chunk 4 ks + u
  //   offset = (a_row ^ (ks << 6)) + kb * 16 * ROWB
  const int a_row = r * C::ROWB + ((u ^ swz16_f<C::CPR>(r)) << 4);
  // transposing reads of K: row 32 ks2 + 16 blk + 4 u + (r >> 2), chunk 2 db + ((r & 3) >> 1),
  // second half of the chunk for odd r
  //   offset = (t_row ^ (db << 5)) + (32 ks2 + 16 blk) * ROWB
  const int rl = 4 * u + (r >> 2);
  const int t_row = rl * C::ROWB + ((((r & 3) >> 1) ^ swz16_f<C::CPR>(rl)) << 4) + (r & 1) * 8;

  auto step = [&](int it, const char* kc, const char* vc, char* kn,
                  char* vn) __attribute__((always_inline)) {
    const int j0 = walk.tile * C::BN;
    const int j1 = j0 + C::BN - 1;
    walk.next<!THREE>();
    if (it + 1 < n_tiles) load_tile(walk.tile, kn, vn);
    // (THREE has no scalar registers for the intervals)
    const bool needed = THREE ? wave_valid && j0 <= wb_last.hi && (j1 >= wb_first.lo || j0 < a.n_sink)
                              : (unsigned)(j0 - need_lo) < need_n || j0 < need_sink;
    if (needed) {
      const bool full = THREE ? wave_rows_full && j1 <= wb_first.hi && (j0 >= wb_last.lo || j1 < a.n_sink)
                              : (unsigned)(j0 - wb_last.lo) < full_n || j0 < full_sink;
      // S^T and dP^T (element i of tile [kb][qb]: key 16 kb + 4 u + i, query 16 qb + r); every
      // K / V fragment read feeds the MFMAs of both query blocks; the chains start from the
      // row statistics.  The two waves of a SIMD overlap best when each keeps its matrix and
      // its vector work apart: vector instructions placed between a wave's own MFMAs hold its
      // MFMAs back, the other wave's do not.
      f32x4 sacc[KBLK][2], pacc[KBLK][2];
      // (the lane offset is made opaque here: its XOR variants, times the buffers, would
      // otherwise be kept in registers across the whole loop)
      int a_off = a_row;
      asm volatile("" : "+v"(a_off));
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int kb = 0; kb < KBLK; kb++) {
          const int off = (a_off ^ (ks << 6)) + kb * 16 * C::ROWB;
          const V8 kfrag = *(const V8*)(kc + off);
          const V8 vfrag = *(const V8*)(vc + off);
#pragma unroll
          for (int qb = 0; qb < 2; qb++) {
            sacc[kb][qb] = M::mfma16(kfrag, qf[qb][ks], ks == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sacc[kb][qb]);
            pacc[kb][qb] = M::mfma16(vfrag, dof[qb][ks], ks == 0 ? delta[qb] : pacc[kb][qb]);
          }
        }
      {
        constexpr int NRD = 2 * KBLK * KS, AH = THREE ? 3 : RSWA_DQ_AH1;  // LDS reads AH ahead, 2 MFMAs each
        __builtin_amdgcn_sched_group_barrier(0x100, AH, 0);
#pragma unroll
        for (int i = 0; i < NRD - AH; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * AH, 0);
      }
      // P = exp2(S c - lse2), dS^T = P (dP^T - delta), packed slab by slab (32 keys) as the B
      // operands of dQ^T += K^T dS^T
#pragma unroll
      for (int kb = 0; kb < KBLK; kb++)
#pragma unroll
        for (int qb = 0; qb < 2; qb++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            sacc[kb][qb][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][qb][i], a.scale_log2, lse2[qb])) *
                              pacc[kb][qb][i];
      if (!full) {
        // edge tile: key j = j0 + 16 kb + i + 4 u is visible iff j <= hi and (j >= lo or j < n_sink); a
        // comparison with a constant and a select per score for the bound that cuts the tile (us, dQ with
        // statistics, before / after: 4001 rows, window 1024 91.5 / 89.3; the pack of short sequences
        // 180 / 176).  The lane's own bounds are recomputed here: kept across the loop they would cost
        // registers.
        int lane_m = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(lane_m));
        const int at = j0 + 4 * (lane_m >> 4);
        int hi_rel[2], lo_rel[2];
#pragma unroll
        for (int qb = 0; qb < 2; qb++) {
          const RowBounds rb = row_bounds(a, r0 + 16 * qb + (lane_m & 15), len_q, len_k);
          hi_rel[qb] = rb.hi - at;
          lo_rel[qb] = rb.lo - at;
        }
        auto keep = [&](auto visible) __attribute__((always_inline)) {
#pragma unroll
          for (int kb = 0; kb < KBLK; kb++)
#pragma unroll
            for (int qb = 0; qb < 2; qb++)
#pragma unroll
              for (int i = 0; i < 4; i++)
                sacc[kb][qb][i] = visible(16 * kb + i, qb) ? sacc[kb][qb][i] : 0.f;
        };
        if (THREE ? !(wave_rows_full && j1 <= wb_first.hi) : j0 >= full_end) keep([&](int c, int qb) { return c <= hi_rel[qb]; });
        if (j0 < wb_last.lo && j1 >= a.n_sink) {
          if (j0 < a.n_sink) {  // some of the tile's keys are sinks
            const int sink_rel = a.n_sink - at;
            keep([&](int c, int qb) { return (c >= lo_rel[qb]) | (c < sink_rel); });
          } else {
            keep([&](int c, int qb) { return c >= lo_rel[qb]; });
          }
        }
      }
      V8 dsb[2][2];
#pragma unroll
      for (int ks2 = 0; ks2 < 2; ks2++)
#pragma unroll
        for (int qb = 0; qb < 2; qb++) {
          float dsv[8];
#pragma unroll
          for (int e = 0; e < 8; e++) dsv[e] = sacc[2 * ks2 + (e >> 2)][qb][e & 3];
          dsb[ks2][qb] = M::pack(dsv);
          asm volatile("" : "+v"(dsb[ks2][qb]));
        }
      int t_off = t_row;
      asm volatile("" : "+v"(t_off));
#pragma unroll
      for (int ks2 = 0; ks2 < 2; ks2++)
#pragma unroll
        for (int d = 0; d < DB; d++) {
          const int off = (t_off ^ (d << 5)) + ks2 * 32 * C::ROWB;
          const V8 kt = tr_pair<V8>(kc + off, kc + off + 16 * C::ROWB);
#pragma unroll
          for (int qb = 0; qb < 2; qb++) dq_acc[d][qb] = M::mfma16(kt, dsb[ks2][qb], dq_acc[d][qb]);
        }
      {
        constexpr int NFR = 2 * DB, AH = THREE ? 2 : RSWA_DQ_AH2;  // transposed fragments (2 reads, 2 MFMAs each)
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * AH, 0);
#pragma unroll
        for (int i = 0; i < NFR - AH; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * AH, 0);
      }
    }
    __syncthreads();
  };

  __syncthreads();
  for (int it = 0; it < n_tiles; it += 2) {
    step(it, k_s0, v_s0, k_s1, v_s1);
    if (it + 1 < n_tiles) step(it + 1, k_s1, v_s1, k_s0, v_s0);
  }

  // ---- epilogue: dq = scale * acc, transposed through LDS for 16-byte stores ------
  // element i of dq_acc[d][qb] is dQ[query 16 qb + r][16 d + 4 u + i]
  char* stage = (wave & 3) == 0 ? k_s0 : (wave & 3) == 1 ? k_s1 : (wave & 3) == 2 ? v_s0 : v_s1;
  for (int half = 0; half < NW / 4; half++) {
    if ((wave >> 2) == half) {
#pragma unroll
      for (int d = 0; d < DB; d++)
#pragma unroll
        for (int qb = 0; qb < 2; qb++) {
          const auto h4 = M::pack4(dq_acc[d][qb][0] * a.scale, dq_acc[d][qb][1] * a.scale,
                                   dq_acc[d][qb][2] * a.scale, dq_acc[d][qb][3] * a.scale);
          *(typename M::V4*)(stage + (16 * qb + r) * C::O_STRIDE + (16 * d + 4 * u) * 2) = h4;
        }
    }
    __syncthreads();
    if ((wave >> 2) == half) {
      constexpr int RPI = 64 / C::CPR;
      const int row0 = lane / C::CPR, col = (lane % C::CPR) * 8;
      const char* src = stage + row0 * C::O_STRIDE + col * 2;
      put_rows<T, RPI, 32 / RPI>(a.dq, dq_off + (int64_t)(r0 + row0) * a.dq_st[1] + col, a.dq_st[1],
                                 len_q - r0 - row0, wave_rows_full, a.wide_dq, a.dq_accumulate,
                                 [&](int n) { return *(const V8*)(src + n * RPI * C::O_STRIDE); });
    }
    __syncthreads();
  }
}

// ============================================================================
// dQ from handed-over dS
// ============================================================================
// The dK/dV kernel of the hand-off route leaves, per (q head, 32-row query tile, 64-key group),
// the 16-bit dS values it computed (zero where the mask hides a pair): a 4 KiB unit of four
// 1 KiB pieces [32-key block kb][query half ks2], a piece holding for each of its 32 keys 32
// bytes: the key's dS for queries 16 ks2 + {0..3, 8..11} and then 16 ks2 + {4..7, 12..15}.  This
// kernel only computes dQ^T += K^T dS^T (2 D multiply-adds per pair, against the 6 D of the
// kernel that recomputes S and dP), so it is bound by reading those units once: it keeps two
// stages of them in flight while it works on a third.
//
// Block = 4 waves; a wave owns 64 query rows (two 32-row tiles) of one q head: the 4 waves are
// 4 / 2 / 1 q heads of a GQA group on the same 64 / 128 / 256 rows, sharing each 64-key K tile.
// Per 16 keys and wave: A = K^T (32 d x 16 keys, transposing reads of the K tile), B = dS^T
// (16 keys x 32 queries, transposing reads of the unit: the 16-lane groups of such a read take
// 4 keys x 16 queries, which is 128 consecutive bytes of a piece), C = dQ^T (lane = query).
template <int D>
struct DqDsCfg {
  static constexpr int BN = 64;   // keys per stage
  static constexpr int NST = 3;   // stages held in LDS
  static constexpr int ROWB = D * 2;
  static constexpr int CPR = D / 8;
  static constexpr int DBLK = D / 32;
  static constexpr int K_TILE = BN * ROWB;
  // LDS image of a unit: piece (kb, ks2) at kb KBLK + ks2 PIECE1 -- 128 bytes between the two
  // query halves, which the two halves of a half-wave read together, put them on different banks
  static constexpr int PIECE1 = 1024 + 128;
  static constexpr int KBLK = 2048 + 256;
  static constexpr int UNIT_LDS = 2 * KBLK;
  static constexpr int WAVE_LDS = 2 * UNIT_LDS;
  static constexpr int O_STRIDE = D * 2 + 16;
  static_assert(WAVE_LDS >= 32 * O_STRIDE, "a wave's epilogue staging fits its dS buffers of a stage");
  static constexpr int NKD = BN * CPR / 256;  // K tile load instructions per wave and stage
  static constexpr int NLD = NKD + 8;         // ... and all loads
};

template <typename T, int D>
__global__ __launch_bounds__(256) void attn_bwd_dq_ds_kernel(const AttnArgs a) {
  using C = DqDsCfg<D>;
  using M = Mma<T>;
  using V8 = typename M::V8;
  constexpr int DB = C::DBLK;
  __shared__ __attribute__((aligned(1024))) char k_s0[C::K_TILE];
  __shared__ __attribute__((aligned(1024))) char k_s1[C::K_TILE];
  __shared__ __attribute__((aligned(1024))) char k_s2[C::K_TILE];
  __shared__ __attribute__((aligned(1024))) char ds_s0[4 * C::WAVE_LDS];
  __shared__ __attribute__((aligned(1024))) char ds_s1[4 * C::WAVE_LDS];
  __shared__ __attribute__((aligned(1024))) char ds_s2[4 * C::WAVE_LDS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c32 = lane & 31;  // query column of a tile
  const int gg = lane >> 5;   // k half
  const int i16 = lane & 15;

  // heads per block: 4, 2 or 1 (the rest of the waves go to further 64-row units)
  const int hsh = (a.group & 3) == 0 ? 2 : (a.group & 1) == 0 ? 1 : 0;
  const int units = a.group >> hsh;
  const int bm_log2 = 8 - hsh;  // 64 rows x (4 >> hsh) units
  const int bm = 1 << bm_log2;
  int rest, hu;
  if (!tile_of_block(a, units, rest, hu)) return;
  const int slot = a.rev_q ? a.n_tile - 1 - rest % a.n_tile : rest % a.n_tile;
  rest /= a.n_tile;
  const int hk = rest % a.heads_kv;
  const int hq = hk * a.group + (hu << hsh) + (wave & ((1 << hsh) - 1));
  SeqInfo s;
  int qt;
  if (a.cu_q) {
    if (!locate_packed(a, slot, bm_log2, false, s, qt)) return;
  } else {
    s.batch_idx = rest / a.heads_kv;
    s.q_row0 = s.k_row0 = 0;
    s.len_q = a.seqlen_q;
    s.len_k = a.seqlen_k;
    qt = slot;
  }
  const int b = s.batch_idx;
  const int len_q = s.len_q, len_k = s.len_k;
  const int i0 = qt << bm_log2;
  if (i0 >= len_q) return;

  const T* k_ptr = (const T*)a.k + b * a.k_st[0] + s.k_row0 * a.k_st[1] + hk * a.k_st[2];
  const T* k2_ptr = a.k2 ? (const T*)a.k2 + b * a.k_st[0] + hk * a.k_st[2] : k_ptr;
  const int64_t dq_off = b * a.dq_st[0] + s.q_row0 * a.dq_st[1] + hq * a.dq_st[2];  // (T or fp32)

  // ---- key stages of the block (64 keys each): those any of its rows can see -------------
  const int i_last = min(i0 + bm, len_q) - 1;
  const int lo_blk = row_bounds(a, i0, len_q, len_k).lo;
  const int hi_blk = row_bounds(a, i_last, len_q, len_k).hi;
  const int t_lo = lo_blk / C::BN;
  const int n_st = hi_blk >= lo_blk ? hi_blk / C::BN - t_lo + 1 : 0;

  // ---- this wave's two row tiles, and for which stages j0 the dK/dV kernel wrote their unit:
  // its wave (keys j0 .. j0 + 63) computed tile i iff some pair of the two survives the mask,
  //   i < len_q, j0 < len_k, j0 <= min(i + 31, len_q - 1) + shift + right,
  //   min(j0 + 63, len_k - 1) >= i + shift - left
  const int r0 = i0 + ((wave >> hsh) << 6);
  const int shift = a.shift_explicit ? a.shift_val : len_k - len_q;
  constexpr int kInf = 1 << 30;
  int jmin[2], jmax[2];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int it = r0 + 32 * t;
    jmax[t] = (a.wr < 0) ? len_k - 1 : min(len_k - 1, min(it + 31, len_q - 1) + shift + a.wr);
    jmin[t] = (a.wl < 0) ? -kInf : it + shift - a.wl - (C::BN - 1);
    if (it >= len_q || (a.wl >= 0 && it + shift - a.wl > len_k - 1)) jmax[t] = -kInf - 1;
  }

  // ---- the wave's dS units: rows of ds_nkb blocks of 4 units per (head, tile slot) ---------
  const int ds_row_bytes = a.ds_nkb * kDsBlockBytes;
  const int64_t ds_head_bytes = (int64_t)a.ds_slots * ds_row_bytes;
  const int64_t slot0 = a.cu_q ? (s.q_row0 >> 5) + b : (int64_t)b * ((a.seqlen_q + 31) >> 5);
  const int64_t ds_off = hq * ds_head_bytes + (slot0 + (r0 >> 5)) * ds_row_bytes;
  const int64_t ds_left = (int64_t)a.heads_q * ds_head_bytes - ds_off;  // bytes up to the buffer's end
  const int ds_span = r0 < len_q ? (int)min((int64_t)2 * ds_row_bytes, ds_left) : 0;
  const __amdgpu_buffer_rsrc_t ds_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(a.ds + (ds_span > 0 ? ds_off : 0)), 0, ds_span, 0x00020000);
  const int ds_voff = lane * 16;

  TileDma<D, C::BN, 256> k_dma;
  k_dma.init(a.k_st[1], tid);
  const KeyRows<T, C::ROWB, false> k_rows(k_ptr, k2_ptr, a.seg, len_k, a.k_st[1]);

  // load cursor: the stage fetched next
  int ld_j = t_lo * C::BN;
  int ld_kb = (ld_j >> 8) % a.ds_nkb;
  auto load_stage = [&](char* kd, char* dsd) __attribute__((always_inline)) {
    k_dma.load(k_rows.template tile<C::BN>(ld_j), kd);
    const int soff = ld_kb * kDsBlockBytes + ((ld_j >> 6) & 3) * kDsUnitBytes;
    char* dst = dsd + wave * C::WAVE_LDS;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int pc = 0; pc < 4; pc++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            ds_rsrc, (lds_void_t*)(dst + t * C::UNIT_LDS + (pc >> 1) * C::KBLK + (pc & 1) * C::PIECE1), 16,
            ds_voff, t * ds_row_bytes + soff + pc * 1024, 0, 0);
    ld_j += C::BN;
    if ((ld_j & 255) == 0) ld_kb = ld_kb + 1 == a.ds_nkb ? 0 : ld_kb + 1;
  };

  // ---- lane-constant LDS offsets ------------------------------------------------------------
  // transposing reads of K: rows 16 s + 8 gg + (i16 >> 2) (+ 4), chunk 4 db + 2 (c32 / 16) +
  // ((i16 & 3) >> 1), second half of the chunk for odd i16
  //   offset = (kt_row{0,1} ^ (db << 6)) + s * 16 * ROWB
  const int krow = 8 * gg + (i16 >> 2);
  const int kch = 2 * (c32 >> 4) + ((i16 & 3) >> 1);
  const int kt_row0 = krow * C::ROWB + ((kch ^ swz_f<C::CPR>(krow)) << 4) + (i16 & 1) * 8;
  const int kt_row1 = (krow + 4) * C::ROWB + ((kch ^ swz_f<C::CPR>(krow + 4)) << 4) + (i16 & 1) * 8;
  // transposing reads of a dS unit: key 16 (s & 1) + 8 gg + (i16 >> 2) (+ 4) of block s >> 1,
  // queries 16 (c32 / 16) + 4 (i16 & 3) ..: byte (i16 & 1) 16 + ((i16 >> 1) & 1) 8 of the key's 32
  const int ds_row = (c32 >> 4) * C::PIECE1 + krow * 32 + (i16 & 1) * 16 + ((i16 >> 1) & 1) * 8;

  f32x16 acc[2][DB];
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[t][d][i] = 0.f;

  int cur_j = t_lo * C::BN;
  auto stage = [&](int it, const char* kc, const char* dsc, char* kn, char* dsn)
      __attribute__((always_inline)) {
    // this wave's loads of the stage have landed (those of the next one may still fly) ...
    if (it + 1 < n_st) {
      wait_vmem_but<C::NLD>();
    } else {
      wait_vmem_but<0>();
    }
    // ... and everybody's: the K tile is complete, and nobody reads the buffers of the stage
    // before this one any more, which the loads of the stage after the next now overwrite
    lds_barrier();
    if (it + 2 < n_st) load_stage(kn, dsn);
    const int j0 = cur_j;
    cur_j += C::BN;
    const bool n0 = j0 >= jmin[0] && j0 <= jmax[0];
    const bool n1 = j0 >= jmin[1] && j0 <= jmax[1];
    if (!(n0 || n1)) return;
    const char* dsw = dsc + wave * C::WAVE_LDS + ds_row;
    auto body = [&](auto c0, auto c1) __attribute__((always_inline)) {
      constexpr bool T0 = decltype(c0)::value, T1 = decltype(c1)::value;
#pragma unroll
      for (int sl = 0; sl < 4; sl++) {
        V8 kt[DB];
#pragma unroll
        for (int d = 0; d < DB; d++)
          kt[d] = tr_pair<V8>(kc + (kt_row0 ^ (d << 6)) + sl * 16 * C::ROWB,
                              kc + (kt_row1 ^ (d << 6)) + sl * 16 * C::ROWB);
        const int uo = (sl >> 1) * C::KBLK + (sl & 1) * 512;
        if constexpr (T0) {
          const V8 dsf = tr_pair<V8>(dsw + uo, dsw + uo + 128);
#pragma unroll
          for (int d = 0; d < DB; d++) acc[0][d] = M::mfma32(kt[d], dsf, acc[0][d]);
        }
        if constexpr (T1) {
          const V8 dsf = tr_pair<V8>(dsw + C::UNIT_LDS + uo, dsw + C::UNIT_LDS + uo + 128);
#pragma unroll
          for (int d = 0; d < DB; d++) acc[1][d] = M::mfma32(kt[d], dsf, acc[1][d]);
        }
      }
    };
    if (n0 && n1) body(std::true_type{}, std::true_type{});
    else if (n0) body(std::true_type{}, std::false_type{});
    else body(std::false_type{}, std::true_type{});
  };

  if (n_st > 0) load_stage(k_s0, ds_s0);
  if (n_st > 1) load_stage(k_s1, ds_s1);
  for (int it = 0; it < n_st; it += 3) {
    stage(it, k_s0, ds_s0, k_s2, ds_s2);
    if (it + 1 < n_st) stage(it + 1, k_s1, ds_s1, k_s0, ds_s0);
    if (it + 2 < n_st) stage(it + 2, k_s2, ds_s2, k_s1, ds_s1);
  }

  // ---- epilogue: dq = scale * acc, a tile at a time through the wave's own LDS ----------------
  // element i of acc[t][d] is dQ[query 32 t + c32][32 d + 8 (i / 4) + 4 gg + i % 4]
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  char* stg = ds_s0 + wave * C::WAVE_LDS;
#pragma unroll
  for (int t = 0; t < 2; t++) {
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++)
        *(typename M::V4*)(stg + c32 * C::O_STRIDE + (32 * d + 8 * i4 + 4 * gg) * 2) =
            M::pack4(acc[t][d][4 * i4] * a.scale, acc[t][d][4 * i4 + 1] * a.scale,
                     acc[t][d][4 * i4 + 2] * a.scale, acc[t][d][4 * i4 + 3] * a.scale);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int n = 0; n < 32 * C::CPR / 64; n++) {
      const int cc = lane + n * 64;
      const int row = cc / C::CPR, col = (cc % C::CPR) * 8;
      const V8 val = *(const V8*)(stg + row * C::O_STRIDE + col * 2);
      if (r0 + 32 * t + row < len_q)
        put_grad8<T>(a.dq, dq_off + (int64_t)(r0 + 32 * t + row) * a.dq_st[1] + col, val, a.wide_dq,
                     a.dq_accumulate);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// ============================================================================
// row statistics, stored negated: -delta = -sum_d dO * O and -lse2 = -lse * log2(e) (empty
// rows: -inf, so that P = exp2(S*c - lse2) is zero).  One 16-lane (D=128) or 8-lane (D=64) group per
// (row, head).
// ============================================================================
// A block owns PrepCfg::ROWS consecutive rows of one q head -- the statistics, [head][row], are then
// written as whole cache lines -- and neighbouring blocks take neighbouring heads, so that the
// blocks in flight sweep out / dout as one dense front; all eight loads of a thread's four rows
// are issued before the first use (one row per thread and the heads innermost: 39 -> 27 us on
// 8192 rows x 32 heads, head_dim 128).
template <int D>
struct PrepCfg {
  static constexpr int LPR = D / 8;         // lanes per row
  static constexpr int RP = 256 / LPR;      // rows per pass
  static constexpr int NR = 4;              // passes
  static constexpr int ROWS = RP * NR;      // rows per block
};

template <typename T, int D>
__global__ __launch_bounds__(256) void attn_bwd_prep_kernel(const AttnArgs a) {
  using P = PrepCfg<D>;
  using V8 = typename Mma<T>::V8;
  // arrival counters of the sink kernel start from zero
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n_count; i += (int64_t)gridDim.x * 256)
    a.sink_count[i] = 0;
  // The delta array starts at the next 256-byte boundary after the lse2 array, and the tile
  // kernels read up to a tile of rows past the last one as statistics: the elements in between
  // get the neutral value (P exactly zero) rather than whatever the workspace held.
  if (blockIdx.x == 0) {
    const int64_t used = a.rows_q * a.heads_q;
    if (used + threadIdx.x < a.delta - a.lse2) a.lse2[used + threadIdx.x] = -__builtin_inff();
  }
  // the first block of a pack's launch writes the key tile table
  if (a.ktile && blockIdx.x == 0) {
    __shared__ int wave_sum[4];
    write_ktile<256>(a, wave_sum);
    return;
  }
  const unsigned blk = blockIdx.x - (a.ktile ? 1 : 0);
  const int h = (int)(blk % (unsigned)a.heads_q);
  const int64_t row0 = (int64_t)(blk / (unsigned)a.heads_q) * P::ROWS + threadIdx.x / P::LPR;
  const int c = (threadIdx.x % P::LPR) * 8;
  // Packed rows past the last sequence belong to nobody: their out / dout may hold anything
  // (NaN included), and the tile kernels read the statistics of the rows that follow a
  // sequence's last tile.  They get the neutral pair, which keeps P and dS exactly zero.
  const int64_t rows_real = a.cu_q ? (int64_t)a.cu_q[a.batch] : a.rows_q;
  V8 o8[P::NR], d8[P::NR];
  float l[P::NR];
#pragma unroll
  for (int i = 0; i < P::NR; i++) {
    const int64_t row = row0 + i * P::RP;
    o8[i] = d8[i] = V8{0, 0, 0, 0, 0, 0, 0, 0};
    l[i] = -__builtin_inff();
    if (row < rows_real) {
      int64_t o_off, do_off, l_off;
      if (a.cu_q) {
        o_off = row * a.o_st[1];
        do_off = row * a.do_st[1];
        l_off = row * a.lse_st[2];
      } else {
        const int64_t bb = row / a.seqlen_q, ii = row % a.seqlen_q;
        o_off = bb * a.o_st[0] + ii * a.o_st[1];
        do_off = bb * a.do_st[0] + ii * a.do_st[1];
        l_off = bb * a.lse_st[0] + ii * a.lse_st[2];
      }
      o8[i] = *(const V8*)((const T*)a.out + o_off + h * a.o_st[2] + c);
      d8[i] = *(const V8*)((const T*)a.dout + do_off + h * a.do_st[2] + c);
      if (c == 0) l[i] = a.lse[l_off + h * a.lse_st[1]];
    }
  }
#pragma unroll
  for (int i = 0; i < P::NR; i++) {
    const int64_t row = row0 + i * P::RP;
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) acc += (float)o8[i][j] * (float)d8[i][j];
#pragma unroll
    for (int m = P::LPR / 2; m >= 1; m >>= 1) acc += __shfl_xor(acc, m, 64);
    if (c == 0 && row < a.rows_q) {
      a.delta[(int64_t)h * a.rows_q + row] = -acc;  // (rows nobody owns: -0)
      a.lse2[(int64_t)h * a.rows_q + row] = (l[i] == -__builtin_inff()) ? l[i] : -l[i] * kLog2e;
    }
  }
}

// Explicit instantiations: with implicit instantiation alone this hipcc emits the host
// launch stubs of only some of the variants.
#define RSWA_INSTANTIATE(T, D)                                              \
  template __global__ void attn_bwd_dkdv_kernel<T, D, false, false, false>(const AttnArgs); \
  template __global__ void attn_bwd_dkdv_kernel<T, D, false, false, true>(const AttnArgs); \
  template __global__ void attn_bwd_dkdv_kernel<T, D, true, false, false>(const AttnArgs); \
  template __global__ void attn_bwd_dkdv_kernel<T, D, true, false, true>(const AttnArgs); \
  template __global__ void attn_bwd_dkdv_kernel<T, D, false, true, false>(const AttnArgs); \
  template __global__ void attn_bwd_dkdv_kernel<T, D, false, true, true>(const AttnArgs); \
  template __global__ void attn_bwd_dq_ds_kernel<T, D>(const AttnArgs);                     \
  template __global__ void attn_bwd_dq_kernel<T, D, false, 4, false>(const AttnArgs); \
  template __global__ void attn_bwd_dq_kernel<T, D, false, 4, true>(const AttnArgs); \
  template __global__ void attn_bwd_dq_kernel<T, D, true, 4, false>(const AttnArgs); \
  template __global__ void attn_bwd_sink_kernel<T, D, 1>(const AttnArgs);               \
  template __global__ void attn_bwd_sink_kernel<T, D, 2>(const AttnArgs);               \
  template __global__ void attn_bwd_prep_kernel<T, D>(const AttnArgs);
RSWA_INSTANTIATE(__bf16, 128)
RSWA_INSTANTIATE(__bf16, 64)
RSWA_INSTANTIATE(_Float16, 128)
RSWA_INSTANTIATE(_Float16, 64)
#undef RSWA_INSTANTIATE
#define RSWA_INSTANTIATE(T)                                                           \
  template __global__ void attn_bwd_dq_kernel<T, 128, false, 8, false>(const AttnArgs); \
  template __global__ void attn_bwd_dq_kernel<T, 128, false, 8, true>(const AttnArgs); \
  template __global__ void attn_bwd_dq_kernel<T, 128, true, 8, false>(const AttnArgs);
RSWA_INSTANTIATE(__bf16)
RSWA_INSTANTIATE(_Float16)
#undef RSWA_INSTANTIATE

// Does the dK/dV launch take blocks of 64 keys whose waves share out the walk (WALK4) instead of
// blocks of 256 keys?  Both forms keep every compute unit busy with one block; what decides is how
// evenly the launch's blocks fill the chip.  Estimated time of a form = the larger of its longest
// block and of rounds x average block, a block being steps x (time of a step) + (prologue and
// epilogue), with times fitted to launches of all kinds (us): head_dim 128, 1.2 + 20 wide, 1.5 + 10 WALK4;
// head_dim 64, 0.77 + 18 and 0.93 + 7.  (A round of equal blocks on every compute unit, whose clock is
// lower, measures 1.58 + 15 and 1.77 + 8.5, 0.91 + 9 and 0.98 + 7.4, which choose no better: 0.4 % behind
// the better form where these are 0.35 %, see below.)  Measured on both sides of the line (us, wide / WALK4, bf16,
// head_dim 128): 32 / 8 heads, window 1024, 4096 rows 217 / 128, 6000 rows 218 / 190, 8192 rows (256
// wide blocks, one full round) 229 / 255, 9000 rows 368 / 303, 16384 rows 477 / 523; 32 / 32 heads,
// window 1000, 2 x 8192 rows 545 / 700; 4096 rows, 32 / 8 heads, causal without a window 623 / 252, without
// a mask 620 / 454.  Of 178 dense and packed shapes drawn, with grouped heads or with at most a round of wide
// blocks, the rule is 0.35 % behind the better form on average (more than 3 % on 6 of them, 14 % at most).
// A pack is judged on its average length L, the only one the host knows, as if of sequences of
// 1.5 L (what a token sees when lengths vary), the longest as long as the pack or the window, with
// half a key tile per sequence wasted.  Packs of 16384 tokens, 32 / 8 heads, window 1024, lengths log-uniform: 16-64
// 262 / 173, 64-256 193 / 175, 16-1024 260 / 216; all of 512 198 / 204, 32 / 32 heads 16-1024 348 / 475.
// The 0.9 leans to the wide form where lengths are alike (65536 tokens of 512: 715 / 784).
bool dkv_walk4(const AttnArgs& a, int head_dim) {
  if (a.dkdv_form == RSWA_DKDV_WIDE || a.dkdv_form == RSWA_DKDV_SHORT) return a.dkdv_form == RSWA_DKDV_SHORT;
  const bool pack = a.cu_q != nullptr;
  const int64_t lk1 = pack ? std::max<int64_t>(1, a.rows_k / a.batch) : a.seqlen_k;
  // As many kv heads as q heads: a walk has no heads to deal, only query tiles, and with clearly more than
  // a round of 256-key blocks the short form loses by its longer fetches (us, wide / short, bf16, head_dim
  // 128: a pack of 3010 tokens, 32 heads, window 2028, 54 / 96; 31427 tokens, 4 heads, 715, 133 / 164;
  // dense 7428 rows, 12 heads, 64, 58 / 70).  Up to 1.25 rounds the estimate decides.  Of 335 such shapes drawn
  // its choice is 2 % behind the better form on average, wide blocks alone 12 % (a pack of 7408 tokens, 8 heads,
  // window 1374, 83 / 62; 8061 tokens, 8 heads, causal, 137 / 88); but it misses where a second round is hardly
  // filled, which a pack's average length does not show: on 43 of them it is 3 % slower than wide blocks or more,
  // by 41 % at most (18 sequences of 213 tokens, 12 heads, head_dim 64, 21.5 / 29.5; 4 of 1991, 8 heads, window
  // 174, 39 / 51).  Staying wide where ceil(average / 256) tiles per sequence fit one round cured those and
  // lost as much elsewhere (2.7 % behind on 260 fresh shapes, 1.8 % without).  Beyond 1.25 rounds WALK4 took 25 %
  // less to 35 % more, 2 % less on average of 67 shapes.
  const double wide_tiles = pack ? (double)lk1 / kDkvKeysPerBlock + 0.5 : (double)ceil_div(lk1, kDkvKeysPerBlock);
  if (a.group == 1 && wide_tiles * a.heads_kv * a.batch > 1.25 * kComputeUnits) return false;
  const int64_t lq1 = pack ? std::max<int64_t>(1, a.rows_q / a.batch) : a.seqlen_q;
  const int64_t lq = pack ? std::min(a.rows_q, lq1 * 3 / 2) : lq1, lk = pack ? std::min(a.rows_k, lk1 * 3 / 2) : lk1;
  // query rows that see a key, of the first the band kernel owns to the last: on average, at most
  const int64_t sh = a.shift_explicit ? a.shift_val : lk - lq;
  const int64_t first = a.wl >= 0 ? std::min<int64_t>(a.n_sink, std::max<int64_t>(lk - 1, 0)) : 0;
  double avg_rows = 0, max_rows = 0;
  for (int t = 0; t <= 16; t++) {
    const int64_t j = std::max((lk - 1) * t / 16, first);
    const int64_t lo = a.wr >= 0 ? std::max<int64_t>(0, j - sh - a.wr) : 0;
    const int64_t hi = a.wl >= 0 ? std::min(lq - 1, j - sh + a.wl) : lq - 1;
    const double r = (double)std::max<int64_t>(0, hi - lo + 1);
    avg_rows += r / 17;
    max_rows = std::max(max_rows, r);
  }
  if (pack) {
    max_rows = (double)a.rows_q;
    if (a.wl >= 0 && a.wr >= 0) max_rows = std::min(max_rows, (double)a.wl + a.wr + 1);
  }
  auto estimate = [&](int keys, int walkers, double step, double fixed) {
    auto walk = [&](double rows, int64_t len) {  // steps of a wave whose keys are seen by `rows` rows each
      const double r = std::min<double>((double)len, rows + (double)std::min<int64_t>(keys, lk1) - 1);
      return std::max(a.group * r / (32. * walkers), std::ceil((double)a.group / walkers));
    };
    const double avg = walk(avg_rows, lq), most = walk(max_rows, pack ? a.rows_q : lq);
    const double tiles = pack ? (double)lk1 / keys + 0.5 : (double)ceil_div(lk1, keys);
    double rounds = tiles * a.heads_kv * a.batch / kComputeUnits;
    // (blocks of equal length run in whole rounds; those of a ramp fill each other's gaps)
    if (rounds < 4 && avg > 0.7 * most) rounds = std::ceil(rounds);
    return std::max(most * step + fixed, rounds * (avg * step + fixed));
  };
  const double lean = pack ? 0.9 : 1.;
  return head_dim == 128 ? estimate(64, 4, 1.5, 10.) < lean * estimate(256, 1, 1.2, 20.)
                         : estimate(64, 4, 0.93, 7.) < lean * estimate(256, 1, 0.77, 18.);
}

template <typename T, int D>
int launch_bwd(AttnArgs& a, hipStream_t stream, int phases) {
  const int64_t units = a.rows_q * a.heads_q;
  const bool walk4 = dkv_walk4(a, D);
  a.ktile_log2 = walk4 ? 6 : 8;
  if (!(phases & RSWA_BWD_DKDV)) a.ktile = nullptr;  // the table serves the dK/dV launch of its own call
  auto launch_dq = [&](auto stats) {
    constexpr bool STATS = decltype(stats)::value;
    const bool pair = (a.group & 1) == 0;
    const bool small = D == 64 || a.avg_keys <= RSWA_DQ_SMALL_AVG_KEYS;
    const int bm = (pair ? 16 : 32) * (small ? 4 : 8);
    a.n_tile = (int)(a.cu_q ? ceil_div(a.rows_q, bm) + a.batch : ceil_div(a.seqlen_q, bm));
    if (a.n_tile == 0) return (int)RSWA_OK;
    const int64_t blocks = deal_blocks(a, pair ? a.group / 2 : a.group, spread_rows(a));
    // (rows a block may have with this window, whatever the call's lengths: no more keys a row, no block of 256)
    const bool never_large = D == 64 || (int64_t)a.wl + a.wr + 1 + a.n_sink <= RSWA_DQ_SMALL_AVG_KEYS;
    a.by_walk = walk_period(a, never_large ? 128 : 256, DqCfg<D>::BN);
    clear_launch_error();
    const dim3 grid((unsigned)blocks), block(small ? 256 : 512);
    if constexpr (!STATS) {
      if (a.far) {
        if (small) {
          hipLaunchKernelGGL((attn_bwd_dq_kernel<T, D, true, 4, false>), grid, block, 0, stream, a);
        } else {
          if constexpr (D == 128) hipLaunchKernelGGL((attn_bwd_dq_kernel<T, D, true, 8, false>), grid, block, 0, stream, a);
        }
        return check_launch("attn_bwd dq");
      }
    }
    if (small) {
      hipLaunchKernelGGL((attn_bwd_dq_kernel<T, D, false, 4, STATS>), grid, block, 0, stream, a);
    } else {
      if constexpr (D == 128) hipLaunchKernelGGL((attn_bwd_dq_kernel<T, D, false, 8, STATS>), grid, block, 0, stream, a);
    }
    return check_launch("attn_bwd dq");
  };
  // Statistics and dQ asked for in one call: the dQ kernel goes first and makes the statistics.
  // (dS hand-off: dQ needs the dK/dV kernel's tiles, so the statistics have a kernel of their own;
  // so they have where the dQ kernel would spill, in the second addressing form, and where dq lies
  // over an input, which dK/dV have to read before it is written.)
  const bool fused = units > 0 && (phases & RSWA_BWD_PREP) && (phases & RSWA_BWD_DQ) && !a.ds && !a.far && !a.dq_last;
  if (fused) {
    if (a.cu_q || a.n_count > 0) {
      clear_launch_error();
      hipLaunchKernelGGL(attn_bwd_rest_kernel, dim3(1), dim3(256), 0, stream, a);
      int rc = check_launch("attn_bwd rest");
      if (rc != RSWA_OK) return rc;
    }
    int rc = launch_dq(std::true_type{});
    if (rc != RSWA_OK) return rc;
  } else if (units > 0 && (phases & RSWA_BWD_PREP)) {
    const int64_t blocks = ceil_div(a.rows_q, PrepCfg<D>::ROWS) * a.heads_q + (a.ktile ? 1 : 0);
    RSWA_REQUIRE(blocks < (1ll << 31), RSWA_ERR_UNSUPPORTED, "attn_bwd: too many (row, head) pairs");
    clear_launch_error();
    hipLaunchKernelGGL((attn_bwd_prep_kernel<T, D>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
    int rc = check_launch("attn_bwd prep");
    if (rc != RSWA_OK) return rc;
  }
  if (phases & RSWA_BWD_DKDV) {
    using C = DkvCfg<D>;
    const int bn = walk4 ? C::BN / 4 : C::BN;
    a.n_tile = (int)(a.cu_q ? ceil_div(a.rows_k, bn) + a.batch : ceil_div(a.seqlen_k, bn));
    const int64_t key_blocks = a.n_tile > 0 ? deal_blocks(a, 1, spread_keys(a)) : 0;
    if (a.ktile && !(phases & RSWA_BWD_PREP)) {
      clear_launch_error();
      hipLaunchKernelGGL(attn_bwd_ktile_kernel, dim3(1), dim3(256), 0, stream, a);
      int rc = check_launch("attn_bwd key tile table");
      if (rc != RSWA_OK) return rc;
    }
    // (an XCD that takes every second tile meets the same lengths again after half as many)
    const int period = a.n_tile >> std::min<int>(a.xcd_log2, __builtin_ctz(a.n_tile | 8));
    a.snake = !a.cu_q && a.seqlen_k <= kSnakeKeys && (walk4 || period % 4 == 0);
    if (key_blocks > 0) {
      clear_launch_error();
      const dim3 grid((unsigned)key_blocks), block(C::THREADS);
      auto go = [&](auto far, auto hand, auto w4) {
        hipLaunchKernelGGL((attn_bwd_dkdv_kernel<T, D, decltype(far)::value, decltype(hand)::value, decltype(w4)::value>),
                           grid, block, 0, stream, a);
      };
      constexpr std::true_type yes{};
      constexpr std::false_type no{};
      if (a.ds) walk4 ? go(no, yes, yes) : go(no, yes, no);  // (never with a.far: see bwd_layout)
      else if (a.far) walk4 ? go(yes, no, yes) : go(yes, no, no);
      else walk4 ? go(no, no, yes) : go(no, no, no);
      int rc = check_launch("attn_bwd dkdv");
      if (rc != RSWA_OK) return rc;
    }
    if (key_blocks > 0 && a.sink_part && a.rows_q > 0) {
      clear_launch_error();
      const dim3 grid(a.batch * a.heads_kv * a.sink_chunks), block(256);
      if (a.n_sink == 1) hipLaunchKernelGGL((attn_bwd_sink_kernel<T, D, 1>), grid, block, 0, stream, a);
      else hipLaunchKernelGGL((attn_bwd_sink_kernel<T, D, 2>), grid, block, 0, stream, a);
      int rc = check_launch("attn_bwd sink");
      if (rc != RSWA_OK) return rc;
    }
  }
  if ((phases & RSWA_BWD_DQ) && a.ds) {
    const int hsh = (a.group & 3) == 0 ? 2 : (a.group & 1) == 0 ? 1 : 0;
    const int bm = 256 >> hsh;
    a.n_tile = (int)(a.cu_q ? ceil_div(a.rows_q, bm) + a.batch : ceil_div(a.seqlen_q, bm));
    if (a.n_tile > 0) {
      const int64_t blocks = deal_blocks(a, a.group >> hsh, false);
      clear_launch_error();
      hipLaunchKernelGGL((attn_bwd_dq_ds_kernel<T, D>), dim3((unsigned)blocks), dim3(256), 0,
                         stream, a);
      int rc = check_launch("attn_bwd dq (dS hand-off)");
      if (rc != RSWA_OK) return rc;
    }
  } else if ((phases & RSWA_BWD_DQ) && !fused) {
    return launch_dq(std::false_type{});
  }
  return RSWA_OK;
}

}  // namespace
}  // namespace rswa

namespace rswa {
namespace {
int bwd_entry(const rswa_attn_params* p, void* stream, int phases, bool allow_handoff,
              uint64_t max_bytes) {
  AttnArgs a;
  int rc = fill_args(p, true, a, allow_handoff, max_bytes);
  if (rc != RSWA_OK) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (p->dtype == RSWA_BF16) {
    return p->head_dim == 128 ? launch_bwd<__bf16, 128>(a, st, phases)
                              : launch_bwd<__bf16, 64>(a, st, phases);
  }
  return p->head_dim == 128 ? launch_bwd<_Float16, 128>(a, st, phases)
                            : launch_bwd<_Float16, 64>(a, st, phases);
}
}  // namespace
}  // namespace rswa

extern "C" int rswa_attn_bwd_phases(const rswa_attn_params* p, void* stream, int phases) {
  return rswa::bwd_entry(p, stream, phases, true, p ? p->workspace_bytes : 0);
}

extern "C" int rswa_attn_bwd_dkdv_keys(const rswa_attn_params* p) {
  using namespace rswa;
  RSWA_REQUIRE(p != nullptr, RSWA_ERR_INVALID, "attn_bwd: null params");
  rswa_attn_params q = *p;
  q.workspace = (void*)(uintptr_t)256;  // (any aligned address: nothing is launched)
  q.workspace_bytes = ~0ull;
  AttnArgs a;
  const int rc = fill_args(&q, true, a, true);
  if (rc != RSWA_OK) return rc;
  return dkv_walk4(a, p->head_dim) ? kDkvKeysPerBlock / 4 : kDkvKeysPerBlock;
}

extern "C" int rswa_attn_bwd(const rswa_attn_params* p, void* stream) {
  return rswa_attn_bwd_phases(p, stream, RSWA_BWD_PREP | RSWA_BWD_DKDV | RSWA_BWD_DQ);
}

// ---- backward on the library's own statistics buffer --------------------------------------
// The row statistics of rswa_attn_bwd_static live in this array instead of a caller
// workspace.  In host code the array's name is only a handle: its device address is looked
// up once per device (each GPU holds its own copy) and that pointer is what the kernels get.
static __device__ __align__(256) unsigned char scratch[RSWA_BWD_STATIC_MAX_BYTES];

namespace rswa {
namespace {
constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
void* scratch_ptr[kMaxDevices] = {nullptr};

// Device address of `scratch` on the current device (nullptr + error message on failure).
void* scratch_on_current_device() {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    fail(RSWA_ERR_LAUNCH, "attn_bwd_static: hipGetDevice: %s (device %d)", hipGetErrorString(e), dev);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      fail(RSWA_ERR_LAUNCH, "attn_bwd_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
      return nullptr;
    }
    scratch_ptr[dev] = ptr;
  }
  return scratch_ptr[dev];
}
}  // namespace
}  // namespace rswa

extern "C" int rswa_attn_bwd_static_init(void) {
  return rswa::scratch_on_current_device() ? RSWA_OK : RSWA_ERR_LAUNCH;
}

extern "C" int rswa_attn_bwd_static(const rswa_attn_params* p, void* stream) {
  using namespace rswa;
  RSWA_REQUIRE(p != nullptr, RSWA_ERR_INVALID, "attn_bwd_static: null params");
  const uint64_t need = bwd_layout(p, false, RSWA_BWD_STATIC_MAX_BYTES).total_bytes;
  RSWA_REQUIRE(need <= RSWA_BWD_STATIC_MAX_BYTES, RSWA_ERR_UNSUPPORTED,
               "attn_bwd_static: rows * heads_q needs %llu bytes of statistics, the built-in "
               "buffer holds %llu (use rswa_attn_bwd with a caller workspace)",
               (unsigned long long)need, (unsigned long long)RSWA_BWD_STATIC_MAX_BYTES);
  rswa_attn_params q = *p;
  // validate everything else before the device is touched (a placeholder keeps the
  // workspace checks quiet; the real address replaces it below)
  q.workspace = (void*)(uintptr_t)256;
  q.workspace_bytes = RSWA_BWD_STATIC_MAX_BYTES;
  {
    AttnArgs probe;
    int rc = fill_args(&q, true, probe, false, RSWA_BWD_STATIC_MAX_BYTES);
    if (rc != RSWA_OK) return rc;
  }
  void* ptr = scratch_on_current_device();
  if (!ptr) return RSWA_ERR_LAUNCH;
  q.workspace = ptr;
  return bwd_entry(&q, stream, RSWA_BWD_PREP | RSWA_BWD_DKDV | RSWA_BWD_DQ, false,
                   RSWA_BWD_STATIC_MAX_BYTES);
}
