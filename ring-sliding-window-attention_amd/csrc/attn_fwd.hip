// Band / sink attention forward for gfx950: bf16|fp16 MFMA, K/V tiles in LDS,
// online softmax, tiles outside the visible band never touched.
//
// Replaces flash-attn's forward as wrapped at ring_swa/ops/wrap_flash.py:168-273.
//
// One block = 4 waves x 32 query rows sharing every K/V tile it loads: either 64 rows of
// TWO q heads of one GQA group (group size even) or 128 rows of one q head; two blocks (at
// head_dim 64 also three, fwd_three_blocks) fit a compute unit (waves of a SIMD are from independent blocks).  Per 64-key
// tile a wave computes S^T = K Q^T (keys x queries) with v_mfma_f32_32x32x16, so each
// lane owns ONE query column: the row max / sum of the online softmax are in-lane
// reductions plus a single half-wave exchange, and P^T is already laid out as the B
// operand of O^T += V^T P^T.  V^T fragments come straight out of the row-major V tile
// with ds_read_b64_tr_b16.
//
// Pipeline.  K/V tiles are double-buffered in LDS and filled by buffer loads that land
// directly in LDS, issued one (V) and two (K) tiles ahead.  The buffers are SEPARATE
// static __shared__ arrays and the tile loop is unrolled by two, so that every access
// names its buffer statically: only then can the compiler tell that an in-flight load
// does not alias the LDS reads of the current tile, and not wait for it.  The waves of a
// block run in lock-step, one barrier per tile; the softmax of one block runs under the MFMAs
// of the compute unit's other block, and a block's prologue and epilogue under the other's
// tiles.  (An 8-wave block whose two halves ran half a tile apart -- the softmax of one half
// under the MFMAs of the other, two barriers per tile -- measured 5 % slower at window 4096
// and 24 % slower at head_dim 64 and window 1000: half the tile loads per row, but one
// block per compute unit and nothing to cover its prologue and epilogue.)
#include "attn_common.h"

namespace rswa {
namespace {

template <int D>
struct FwdCfg {
  static constexpr int BN = 64;
  static constexpr int THREADS = 256;
  static constexpr int KSTEPS = D / 16;
  static constexpr int DBLK = D / 32;
  static constexpr int CPR = D / 8;   // 16-byte chunks per row
  static constexpr int ROWB = D * 2;  // bytes per row
  static constexpr int TILE = BN * ROWB;
  static constexpr int O_STRIDE = D * 2 + 16;
  static_assert(TILE >= 32 * O_STRIDE, "one wave's epilogue staging fits one tile buffer");
};

// WAVES: blocks per compute unit (a block has one wave per SIMD), see fwd_three_blocks.
template <typename T, int D, bool SKIP, bool FAR, int WAVES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))
void attn_fwd_kernel(const AttnArgs a) {
  using C = FwdCfg<D>;
  constexpr int NW = C::THREADS / 64;
  using M = Mma<T>;
  using V8 = typename M::V8;
  __shared__ __attribute__((aligned(1024))) char k_s0[C::TILE];
  __shared__ __attribute__((aligned(1024))) char k_s1[C::TILE];
  __shared__ __attribute__((aligned(1024))) char v_s0[C::TILE];
  __shared__ __attribute__((aligned(1024))) char v_s1[C::TILE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // (known to be uniform: the rows' bounds are scalars, 20 registers less; with SKIP, whose branches then
  // are scalar ones, the compiler would keep both sides' fragments and spill)
  const int wave = SKIP ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int g = lane >> 5;
  const int i16 = lane & 15;
  const int u = lane >> 4;

  // ---- which (sequence, kv head, q tile, q head(s)) -------------------------
  // pair mode: waves 0-1 and 2-3 take the same 64 rows of two neighbouring q heads;
  // row mode: the 4 waves take 128 consecutive rows of one q head
  const bool pair = (a.group & 1) == 0;
  const int units = pair ? a.group >> 1 : a.group;  // blocks per (kv head, q tile)
  const int bm = pair ? 16 * NW : 32 * NW;          // query rows per block
  int rest, hu;
  if (!tile_of_block(a, units, rest, hu)) return;
  const int tiles_before = quotient(rest, a.by_tile);
  const int tile = rest - tiles_before * a.n_tile;
  const int slot = a.rev_q ? a.n_tile - 1 - tile : tile;
  rest = quotient(tiles_before, a.by_heads);  // batch entry (dense)
  const int hk = tiles_before - rest * a.heads_kv;
  const int hq = hk * a.group + (pair ? 2 * hu + (wave >> 1) : hu);
  SeqInfo s;
  int qt;
  if (a.cu_q) {
    if (!locate_packed(a, slot, pair ? 6 : 7, false, s, qt)) return;
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
  const T* k_ptr = (const T*)a.k + b * a.k_st[0] + s.k_row0 * a.k_st[1] + hk * a.k_st[2];
  const T* v_ptr = (const T*)a.v + b * a.v_st[0] + s.k_row0 * a.v_st[1] + hk * a.v_st[2];
  // (element offsets: out is T or, as a ring accumulator, fp32; lse is fp32 or fp64)
  const int64_t o_off = b * a.o_st[0] + s.q_row0 * a.o_st[1] + hq * a.o_st[2];
  const int64_t lse_off = b * a.lse_st[0] + hq * a.lse_st[1] + s.q_row0 * a.lse_st[2];

  // ---- key tiles this block visits -----------------------------------------
  const int i_last = min(i0 + bm, len_q) - 1;
  const KeyTiles tiles = key_tiles<C::BN>(a, i0, i_last, len_q, len_k);
  const int n_tiles = tiles.n_sink + tiles.n_band;
  KeyWalk walk(a, tiles);
  const int t_first = walk.tile;
  walk.next<false>();

  // ---- this wave's rows ----------------------------------------------------
  const int r0 = i0 + (pair ? wave & 1 : wave) * 32;
  const int iq = r0 + l32;
  const RowBounds rb = row_bounds(a, iq, len_q, len_k);
  const bool wave_rows_full = r0 + 31 < len_q;
  const RowBounds wb_first = row_bounds(a, r0, len_q, len_k);
  const RowBounds wb_last = row_bounds(a, min(r0 + 31, len_q - 1), len_q, len_k);

  // ---- tile DMA: rows past len_k read as zero ---------------------------------
  TileDma<D, C::BN, C::THREADS> k_dma, v_dma;
  k_dma.init(a.k_st[1], tid);
  v_dma.init(a.v_st[1], tid);
  // (keys in two row ranges: the second range's tensors, at this batch entry and kv head)
  const T* k2_ptr = a.k2 ? (const T*)a.k2 + b * a.k_st[0] + hk * a.k_st[2] : k_ptr;
  const T* v2_ptr = a.v2 ? (const T*)a.v2 + b * a.v_st[0] + hk * a.v_st[2] : v_ptr;
  const KeyRows<T, C::ROWB, FAR> k_rows(k_ptr, k2_ptr, a.seg, len_k, a.k_st[1]), v_rows(v_ptr, v2_ptr, a.seg, len_k, a.v_st[1]);
  auto load_k = [&](int tile, char* dst) __attribute__((always_inline)) {
    k_dma.load(k_rows.template tile<C::BN>(tile * C::BN), dst);
  };
  auto load_v = [&](int tile, char* dst) __attribute__((always_inline)) {
    v_dma.load(v_rows.template tile<C::BN>(tile * C::BN), dst);
  };

  // The first tiles and the rows' own data are asked for before anything else is computed: K(0) and Q
  // first, which S(0) needs.  (A block's start and end are 6 of its 31 us at window 1024, 6 of 13 in a
  // pack of short sequences.  This, divisions by multiplication, the search of locate_packed and an
  // epilogue without branches or a 64-bit product per row: us, before / after, 4001 rows, window 1024,
  // 32 / 8 heads 75.4 / 73.0; a pack of 16384 tokens in sequences of 16 to 1024 149 / 144; 2 x 8192 rows,
  // 32 heads, window 1000 358 / 351; 4 x 2000 rows, 28 / 4 heads, head_dim 64, fp16 79.0 / 76.1.)
  if (n_tiles > 0) load_k(t_first, k_s0);
  // Q fragments (B operand of K Q^T): lane = query column, 8 consecutive d per k-step.  (Rows past the
  // end read the last row's values: their columns are masked in every tile and never stored.)
  const T* q_row = q_ptr + (int64_t)min(iq, len_q - 1) * a.q_st[1] + g * 8;
  V8 qf[C::KSTEPS];
#pragma unroll
  for (int ks = 0; ks < C::KSTEPS; ks++) qf[ks] = *(const V8*)(q_row + ks * 16);

  if (n_tiles > 0) load_v(t_first, v_s0);
  if (n_tiles > 1) load_k(walk.tile, k_s1);

  f32x16 o_acc[C::DBLK];
#pragma unroll
  for (int d = 0; d < C::DBLK; d++)
#pragma unroll
    for (int i = 0; i < 16; i++) o_acc[d][i] = 0.f;
  float m_run = -__builtin_inff();  // running max of raw scores (shared by the lane pair)
  float l_run = 0.f;                // this lane's share of the running sum

  // ---- lane-constant LDS offsets (swizzle folded into XOR / immediate parts) ----
  // K row fragments (16-byte reads): row = 32 t + l32, chunk = 2 ks + g
  //   offset = (a_row ^ (ks << 5)) + t * 32 * ROWB
  const int a_row = l32 * C::ROWB + ((g ^ swz_f<C::CPR>(l32)) << 4);
  // transposing reads of V: rows 16 s4 + 4 g + (i16 >> 2) and + 8, chunk = 4 d + lp
  //   offset = (t_row{0,1} ^ (d << 6)) + s4 * 16 * ROWB
  const int rl = 4 * g + (i16 >> 2);
  const int lp = 2 * (u & 1) + ((i16 & 3) >> 1);
  const int t_row0 = rl * C::ROWB + ((lp ^ swz_f<C::CPR>(rl)) << 4) + (i16 & 1) * 8;
  const int t_row1 = (rl + 8) * C::ROWB + ((lp ^ swz_f<C::CPR>(rl + 8)) << 4) + (i16 & 1) * 8;

  // ---- pieces of one tile ------------------------------------------------------
  // S^T[key, query] = K Q^T
  auto qk = [&](const char* kc, f32x16(&sacc)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) sacc[t][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < C::KSTEPS; ks++) {
      const int off = a_row ^ (ks << 5);
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const V8 kf = *(const V8*)(kc + off + t * 32 * C::ROWB);
        sacc[t] = M::mfma32(kf, qf[ks], sacc[t]);
      }
    }
  };
  // mask of an edge tile: visible iff j <= hi and (j >= lo or j < n_sink).  Key j = j0 + c + 4 g, c known
  // per register: either bound is one comparison with a constant and one select per score, and a tile
  // pays for the bound that cuts it.  (As logic on three comparisons for all of it an edge tile had 190
  // instructions more than another, half as many again as the softmax.  us, before / after, with the wave's
  // bounds as scalars: 4001 rows, window 1024, 32 / 8 heads 68.9 / 65.9; a pack of 16384 tokens in
  // sequences of 16 to 1024 140 / 132; 4 x 2000 rows, 28 / 4 heads, head_dim 64, 4 sinks 74.0 / 68.9.)
  auto mask = [&](int tile, f32x16(&sacc)[2]) __attribute__((always_inline)) {
    const int j0 = tile * C::BN;
    const int j1 = j0 + C::BN - 1;
    // score n of the lane: register n % 16 of the tile's 32-key half n / 16
    auto keep = [&](auto visible) __attribute__((always_inline)) {
      select_lanes<32>(
          [&](auto nc) __attribute__((always_inline)) {
            constexpr int n = decltype(nc)::value;
            return visible(n / 16 * 32 + 8 * (n % 16 >> 2) + (n & 3));
          },
          [&](auto nc, bool v) __attribute__((always_inline)) {
            constexpr int t = decltype(nc)::value / 16, i = decltype(nc)::value % 16;
            sacc[t][i] = v ? sacc[t][i] : -__builtin_inff();
          });
    };
    if (!(wave_rows_full && j1 <= wb_first.hi)) {
      const int hi_rel = rb.hi - j0 - 4 * g;
      keep([&](int c) { return lanes(c <= hi_rel); });
    }
    if (j0 < wb_last.lo && j1 >= a.n_sink) {
      int lo_rel = rb.lo - j0 - 4 * g;
      if (j0 < a.n_sink) {  // some of the tile's keys are sinks
        const int sink_rel = a.n_sink - j0 - 4 * g;
        asm volatile("" : "+v"(lo_rel));  // (or both branches' comparisons are made ahead of them, in 64 SGPRs)
        keep([&](int c) { return lanes(c >= lo_rel) | lanes(c < sink_rel); });
      } else {
        keep([&](int c) { return lanes(c >= lo_rel); });
      }
    }
  };
  // online softmax of one tile (raw-score max, exponent in base 2); P^T packed for the
  // PV MFMAs; returns the factor the running output must be scaled by
  auto softmax = [&](f32x16(&sacc)[2], V8(&pb)[4]) __attribute__((always_inline)) -> float {
    float mx = sacc[0][0];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) mx = fmaxf(mx, sacc[t][i]);
    mx = halfwave_max(mx);
    // The reference point of the exponentials moves only when the maximum has grown by
    // more than 2^8: until then P <= 256, exact in fp32 sums and harmless in 16 bits, and
    // the rescale of the running output is skipped for almost every tile.
    const float m_new = fmaxf(m_run, mx);
    const bool bump = (m_new - m_run) * a.scale_log2 > 8.f;  // true from -inf, false for NaN
    const float m_keep = bump ? m_new : m_run;
    const float m_use = (m_keep == -__builtin_inff()) ? 0.f : m_keep;
    // (1 also where the row has seen no key yet: O is zero then, and the first tile needs no rescale)
    const float alpha =
        m_run == -__builtin_inff() ? 1.f : __builtin_amdgcn_exp2f((m_run - m_use) * a.scale_log2);
    const float mc = m_use * a.scale_log2;
    m_run = m_keep;
    float psum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) {
      float pv[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        pv[j] = __builtin_amdgcn_exp2f(
            __builtin_fmaf(sacc[s4 >> 1][8 * (s4 & 1) + j], a.scale_log2, -mc));
        psum[j & 3] += pv[j];
      }
      pb[s4] = M::pack(pv);
      // keep the vector work in the vector phase: the packed P is opaque from here on
      asm volatile("" : "+v"(pb[s4]));
    }
    float psum_all = (psum[0] + psum[1]) + (psum[2] + psum[3]);
    asm volatile("" : "+v"(psum_all));
    l_run = l_run * alpha + psum_all;
    return alpha;
  };
  // O^T[d, query] = alpha * O^T + V^T P^T, in two parts
  auto rescale = [&](float alpha) __attribute__((always_inline)) {
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {
#pragma unroll
      for (int d = 0; d < C::DBLK; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o_acc[d][i] *= alpha;
    }
  };
  auto pv_acc = [&](const char* vc, const V8(&pb)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) {
#pragma unroll
      for (int d = 0; d < C::DBLK; d++) {
        const int off0 = (t_row0 ^ (d << 6)) + s4 * 16 * C::ROWB;
        const int off1 = (t_row1 ^ (d << 6)) + s4 * 16 * C::ROWB;
        o_acc[d] = M::mfma32(tr_pair<V8>(vc + off0, vc + off1), pb[s4], o_acc[d]);
      }
    }
  };

  // ---- tile loop ------------------------------------------------------------------------
  // Per tile: a vector section (mask + softmax of tile t, rescale of O), the block barrier,
  // a matrix section (O += P(t) V(t), S(t+1) = K(t+1) Q^T).  The barrier publishes K(t+1) and
  // V(t), loaded during the previous matrix section, and releases the buffers of K(t) and
  // V(t-1), last read before it: the loads of K(t+2) and V(t+1) into them follow it.
  f32x16 s_cur[2];
  int t_cur = t_first, t_next = walk.tile;  // tiles t and t + 1; the cursor: t + 2
  walk.next<false>();
  auto prefetch = [&](int it, char* kfree, char* vn) __attribute__((always_inline)) {
    if (it + 2 < n_tiles) load_k(walk.tile, kfree);
    if (it + 1 < n_tiles) load_v(t_next, vn);
  };
  // A tile the block visits may hold no key that this wave's 32 rows can see (the block's
  // key range is as wide as the window plus all its rows): the wave then skips the tile's
  // work and only keeps the barrier.  With a short window that is a sizeable share: at
  // window 256 and 128 rows per block a wave needs 5 of the block's 7 tiles.
  // (SKIP is chosen by the host for short windows only: with a long window the test costs
  // more than the rare skipped tile saves.)
  auto wave_needs = [&](int it, int tile) __attribute__((always_inline)) -> bool {
    if constexpr (!SKIP) return it < n_tiles;
    const int j0 = tile * C::BN;
    return it < n_tiles && r0 < len_q && j0 <= wb_last.hi &&
           (j0 + C::BN - 1 >= wb_first.lo || j0 < a.n_sink);
  };
  auto iter = [&](int it, const char* kn, char* kfree, const char* vc,
                  char* vn) __attribute__((always_inline)) {
    // without SKIP both are compile-time true: one path, and after the last tile S(t+1) is
    // computed from stale LDS contents and never used
    const bool need_cur = SKIP ? wave_needs(it, t_cur) : true;
    const bool need_next = SKIP ? wave_needs(it + 1, t_next) : true;
    V8 pb[4];
    if (need_cur) {
      mask(t_cur, s_cur);
      const float alpha = softmax(s_cur, pb);
      rescale(alpha);
    }
    wait_dma();
    lds_barrier();
    if (!(need_cur && need_next)) prefetch(it, kfree, vn);
    if (need_cur && need_next) {
      // matrix section as ONE basic block, LDS reads scheduled four fragments ahead of their
      // MFMA.  The tile loads ride between the MFMAs, one every fourth: issued in a row they
      // hold the wave for about 50 cycles apiece before its first MFMA.  No branch may split
      // the block, so past the last tile some are fetched again, into buffers nobody reads.
      load_k(walk.tile, kfree);
      load_v(t_next, vn);
      pv_acc(vc, pb);
      qk(kn, s_cur);
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
      static_for<32>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (i < 12) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        else if constexpr (i < 28) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if constexpr (i % 4 == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      });
    } else if (need_cur) {
      pv_acc(vc, pb);
    } else if (need_next) {
      qk(kn, s_cur);
    }
    t_cur = t_next;
    t_next = walk.tile;
    walk.next<false>();
  };

  __syncthreads();
  if (wave_needs(0, t_first)) qk(k_s0, s_cur);
  for (int it = 0; it < n_tiles; it += 2) {
    iter(it, k_s1, k_s0, v_s0, v_s1);
    if (it + 1 < n_tiles) iter(it + 1, k_s0, k_s1, v_s1, v_s0);
  }
  __syncthreads();

  // ---- epilogue --------------------------------------------------------------
  const float l_tot = halfwave_sum(l_run);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  // transpose O^T through LDS for coalesced 16-byte stores, one tile buffer per wave
  char* stage = wave == 0 ? k_s0 : wave == 1 ? k_s1 : wave == 2 ? v_s0 : v_s1;
  // out_accumulate: out / lse hold a running partial result; the block is merged into it with
  // the arithmetic of the merge kernel (merge_lse.hip), applied to the block's output after
  // its rounding to 16 bits -- the same bits as a forward into a temporary plus a merge.  The
  // rows' two weights wait in LDS behind the staged tile for the lanes that store the rows.
  float* wgt = (float*)(stage + 32 * C::O_STRIDE);
  static_assert(C::TILE >= 32 * C::O_STRIDE + 32 * 2 * 4, "weights fit behind the staged tile");
  {
    const float ninf = -__builtin_inff();
    float lse_new = l_tot > 0.f ? m_run * a.scale + __logf(l_tot) : ninf;
    float w_old = 0.f, w_new = 1.f;
    const int64_t lse_at = lse_off + (int64_t)iq * a.lse_st[2];
    if (a.out_accumulate && iq < len_q) {
      // (an fp64 running LSE enters the arithmetic as fp32, as in the merge kernel)
      const float la = a.wide_out ? (float)((const double*)a.lse)[lse_at] : a.lse[lse_at];
      const float lb = lse_new;
      const bool both_empty = (la == ninf) && (lb == ninf);
      const float diff = both_empty ? 0.f : lb - la;
      w_old = both_empty ? 0.f : 1.f / (1.f + __expf(diff));
      w_new = both_empty ? 0.f : 1.f / (1.f + __expf(-diff));
      lse_new = both_empty ? ninf : fmaxf(la, lb) + log1pf(__expf(-fabsf(diff)));
    }
    if (g == 0 && iq < len_q) {
      if (a.wide_out) ((double*)a.lse)[lse_at] = (double)lse_new;
      else a.lse[lse_at] = lse_new;
    }
    // (the staging buffer is the wave's own: its writes only have to land before its reads)
#pragma unroll
    for (int d = 0; d < C::DBLK; d++)
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++) {
        const auto h4 = M::pack4(o_acc[d][4 * i4] * inv, o_acc[d][4 * i4 + 1] * inv,
                                 o_acc[d][4 * i4 + 2] * inv, o_acc[d][4 * i4 + 3] * inv);
        *(typename M::V4*)(stage + l32 * C::O_STRIDE + (d * 32 + 8 * i4 + 4 * g) * 2) = h4;
      }
    if (g == 0) {
      wgt[2 * l32] = w_old;
      wgt[2 * l32 + 1] = w_new;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    constexpr int RPI = 64 / C::CPR, N = 32 / RPI;  // rows per store instruction, stores
    const int row0 = lane / C::CPR, col = (lane % C::CPR) * 8;
    const char* src = stage + row0 * C::O_STRIDE + col * 2;
    const int64_t at0 = o_off + (int64_t)(r0 + row0) * a.o_st[1] + col, step = RPI * a.o_st[1];
    const int left = len_q - r0 - row0;  // rows the lane has to store: n RPI < left
    if (!(a.wide_out | a.out_accumulate)) {
      T* dst = (T*)a.out + at0;
      if (wave_rows_full) {
#pragma unroll
        for (int n = 0; n < N; n++) *(V8*)(dst + n * step) = *(const V8*)(src + n * RPI * C::O_STRIDE);
      } else {
#pragma unroll
        for (int n = 0; n < N; n++)
          if (n * RPI < left) *(V8*)(dst + n * step) = *(const V8*)(src + n * RPI * C::O_STRIDE);
      }
      return;
    }
    for (int n = 0; n < N; n++) {
      if (n * RPI < left) {
        V8 val = *(const V8*)(src + n * RPI * C::O_STRIDE);
        const int64_t at = at0 + n * step;
        const int row = row0 + n * RPI;
        const float wo = a.out_accumulate ? wgt[2 * row] : 0.f;
        const float wn = a.out_accumulate ? wgt[2 * row + 1] : 1.f;
        if (a.wide_out) {
          // fp32 accumulator: the block's 16-bit values as fp32, or merged into what it holds
          float* dst = (float*)a.out + at;
          f32x4 y[2];
#pragma unroll
          for (int hh = 0; hh < 2; hh++) {
            f32x4 old = {0.f, 0.f, 0.f, 0.f};
            if (a.out_accumulate) old = *(const f32x4*)(dst + 4 * hh);
#pragma unroll
            for (int j = 0; j < 4; j++) {
              const float t0 = (wo == 0.f) ? 0.f : old[j] * wo;
              const float t1 = (wn == 0.f) ? 0.f : (float)val[4 * hh + j] * wn;
              y[hh][j] = t0 + t1;
            }
          }
          *(f32x4*)dst = y[0];
          *(f32x4*)(dst + 4) = y[1];
        } else {
          T* dst = (T*)a.out + at;
          const V8 old = *(const V8*)dst;
          float y[8];
#pragma unroll
          for (int j = 0; j < 8; j++) {
            // a zero weight must annihilate whatever the other side holds
            const float t0 = (wo == 0.f) ? 0.f : (float)old[j] * wo;
            const float t1 = (wn == 0.f) ? 0.f : (float)val[j] * wn;
            y[j] = t0 + t1;
          }
          *(V8*)dst = M::pack(y);
        }
      }
    }
  }
}

// Explicit instantiations: with implicit instantiation alone this hipcc emits the host
// launch stubs of only some of the four variants.
#define RSWA_INSTANTIATE(T, D, W)                                                   \
  template __global__ void attn_fwd_kernel<T, D, false, false, W>(const AttnArgs); \
  template __global__ void attn_fwd_kernel<T, D, true, false, W>(const AttnArgs);  \
  template __global__ void attn_fwd_kernel<T, D, false, true, W>(const AttnArgs);  \
  template __global__ void attn_fwd_kernel<T, D, true, true, W>(const AttnArgs);
RSWA_INSTANTIATE(__bf16, 128, 2)
RSWA_INSTANTIATE(__bf16, 64, 2)
RSWA_INSTANTIATE(__bf16, 64, 3)
RSWA_INSTANTIATE(_Float16, 128, 2)
RSWA_INSTANTIATE(_Float16, 64, 2)
RSWA_INSTANTIATE(_Float16, 64, 3)
#undef RSWA_INSTANTIATE

int rows_per_block(const AttnArgs& a) { return (a.group & 1) == 0 ? 64 : 128; }
int blocks_per_tile(const AttnArgs& a) { return ((a.group & 1) == 0 ? a.group / 2 : a.group) * a.heads_kv; }

// Three blocks per compute unit instead of two?  head_dim 128 needs 191 registers and 64 KiB of LDS, so two.
// head_dim 64 has half the MFMAs per score and is bound by the softmax's vector work and its latencies;
// it fits three (135 registers, 158 with SKIP; built for four it fits without SKIP and is up to 17 %
// slower).  Three where the launch has more blocks than fit at two per unit (us, two / three: 4 x 2000
// rows, 28 / 4 heads, window 1000, 1792 blocks, 68 / 67; 8192 rows, 32 / 8 heads, window 1024, 91 / 83;
// 2 x 6000 rows, 8 / 2 heads, window 3000, 100 / 81; 2 x 4000 rows, 12 heads, 768 blocks, 60 / 64; where
// they all fit anyway the two are equal), and where blocks are long and of unlike length, so that the
// longest decide, a little over two rounds (causal without a window: 8 heads, 13513 tokens in three
// sequences, 864 blocks, 105 / 121; 32 heads, 2 x 1250 tokens, 640 blocks, 34 / 36; 12 heads, 20738 tokens in
// four, 1968 blocks, 249 / 236).  Between 512 and 1150 uneven blocks either can win, by no rule found (28 / 4
// heads, 3000 tokens, 672 blocks, 69 / 61; 12 heads, 8873 tokens in eleven, 898 blocks, 75 / 66): of 161 shapes
// drawn with 430 to 2600 blocks the rule is 0.8 % behind the better build on average, 14 % at most, three alone
// 0.5 %, two alone 6 %.
bool fwd_three_blocks(const AttnArgs& a, int head_dim) {
  if (head_dim != 64) return false;
  const double tiles = a.cu_q ? (double)a.rows_q / rows_per_block(a) + 0.5 * a.batch
                              : (double)ceil_div(a.seqlen_q, rows_per_block(a)) * a.batch;
  const bool even = a.avg_keys >= 0.7 * a.max_keys || a.avg_keys <= 250;
  return tiles * blocks_per_tile(a) > (even ? 2 * kComputeUnits : 1150);
}

template <typename T, int D, int WAVES>
int launch_fwd(AttnArgs& a, hipStream_t stream) {
  using C = FwdCfg<D>;
  const int bm = rows_per_block(a);
  a.n_tile = (int)(a.cu_q ? ceil_div(a.rows_q, bm) + a.batch : ceil_div(a.seqlen_q, bm));
  if (a.n_tile == 0) return RSWA_OK;
  const int64_t blocks = deal_blocks(a, blocks_per_tile(a) / a.heads_kv, spread_rows(a));
  a.by_walk = walk_period(a, 128, C::BN);
  // keys a row sees at most; the per-wave tile skip pays when the rows of a block beyond one
  // wave's 32 add a tenth or more to that span
  const int64_t span = (a.wl < 0 || a.wr < 0) ? (int64_t)1 << 40 : (int64_t)a.wl + a.wr + 1;
  // (measured at window 1000 and 128-row blocks, where the skip would save a wave one tile in
  // eighteen: no difference either way, 0.435 against 0.431-0.441 ms)
  const bool skip = (bm - 32) * 10 >= span + bm;
  clear_launch_error();
  const dim3 grid((unsigned)blocks), block(C::THREADS);
  if (skip) {
    if (a.far) hipLaunchKernelGGL((attn_fwd_kernel<T, D, true, true, WAVES>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((attn_fwd_kernel<T, D, true, false, WAVES>), grid, block, 0, stream, a);
  } else {
    if (a.far) hipLaunchKernelGGL((attn_fwd_kernel<T, D, false, true, WAVES>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((attn_fwd_kernel<T, D, false, false, WAVES>), grid, block, 0, stream, a);
  }
  return check_launch("attn_fwd");
}

}  // namespace
}  // namespace rswa

extern "C" int rswa_attn_fwd(const rswa_attn_params* p, void* stream) {
  using namespace rswa;
  AttnArgs a;
  int rc = fill_args(p, false, a);
  if (rc != RSWA_OK) return rc;
  if (a.rows_q == 0) return RSWA_OK;
  hipStream_t st = (hipStream_t)stream;
  const bool bf16 = p->dtype == RSWA_BF16;
  if (p->head_dim == 128) return bf16 ? launch_fwd<__bf16, 128, 2>(a, st) : launch_fwd<_Float16, 128, 2>(a, st);
  if (fwd_three_blocks(a, 64)) return bf16 ? launch_fwd<__bf16, 64, 3>(a, st) : launch_fwd<_Float16, 64, 3>(a, st);
  return bf16 ? launch_fwd<__bf16, 64, 2>(a, st) : launch_fwd<_Float16, 64, 2>(a, st);
}

extern "C" int rswa_attn_fwd_blocks_per_cu(const rswa_attn_params* p) {
  using namespace rswa;
  AttnArgs a;
  const int rc = fill_args(p, false, a);
  if (rc != RSWA_OK) return rc;
  return fwd_three_blocks(a, p->head_dim) ? 3 : 2;
}
