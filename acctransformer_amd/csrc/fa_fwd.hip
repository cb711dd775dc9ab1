// FlashAttention2 forward for gfx950 (CDNA4).
//
// Replaces the reference's forward kernel builder
// (train/acctransformer/flash_attention/ops/flash_attention/flash_attention_fwd.py:308-474:
// Q-outer / KV-inner loops, online softmax, O rescale, O/l and L = m + ln l).
//
// Work split: one workgroup (4 or 8 waves) owns 32*QG query rows per wave of one
// (batch, head).  K and V tiles of 64 rows (128 in the variants without side
// inputs) are staged through LDS (double buffered) and shared by the waves.  The wave computes
// the TRANSPOSED score tile S^T = K Q^T with 32x32x16 MFMAs, so every lane
// holds scores of a single query row (column l%32 of the MFMA C tile): the
// online-softmax state (running max, running sum) is per lane, row
// reductions are in-register plus one swap with lane l^32, and the C tile is
// directly the B operand of O^T += V^T P^T.  V^T fragments come from the
// row-major V tile through transposed LDS reads.
#include "fa_common.hpp"
#include "fa_launch.hpp"

#include <type_traits>

#ifndef ACCT_ELEM
#error "compiled once per element type: -DACCT_ELEM=f16 and -DACCT_ELEM=bf16"
#endif

namespace acct {

// LDS of the key-group merge: the accumulators are cut into 4 DB pieces of 8 columns, of which every key group finishes
// 4 DB / KG; a wave leaves the pieces of the other groups here, then its running max and sum.
template <int D, int KG> constexpr int fwd_merge_pieces() { return 4 * SwzCfg<D>::DB / KG; }
template <int D, int NW, int KG> constexpr int fwd_merge_stats() { return NW * (KG - 1) * fwd_merge_pieces<D, KG>() * 1024; }

// Two key groups at head dims up to 64, launches of more than one round: the first group merges alone (see there).
template <int D, int KG> constexpr bool fwd_merge_alone() { return KG == 2 && D <= 64; }

// KG > 1 (small grids): the waves of a workgroup form NW / KG row groups times KG key groups.  A wave then works on
// its key group's share of every tile only, with softmax statistics of its own, and the key groups of a row group
// are merged through LDS before the epilogue -- KG times as many workgroups for the same rows, every wave busy.
template <typename T, int D, int QG, int NW, bool BIAS, bool DROP, bool MASKT, int KT = 2, int KG = 1, bool PIPE = false>
ACCT_DEV void fa_fwd_body(const FaArgs& a) {
  static_assert(KT == 2 || KT == 4 || (KT == 8 && !BIAS && !DROP), "key tiles are 64, 128 or 256 rows (with a bias, 128 rows take the key-only form of it only)");
  static_assert(KG == 1 || (QG == 1 && KT % KG == 0 && NW % KG == 0), "key groups own whole 32-key chunks");
  static_assert(KT / KG <= 4, "a wave's keys of a tile lie in one 128-key block");
  constexpr int BN = 32 * KT;                       // key rows per tile
  constexpr int KTW = KT / KG, WN = 32 * KTW;       // 32-key chunks and keys of a tile that one wave works on
  constexpr int RG = NW / KG;                       // row groups
  static_assert(!PIPE || (!BIAS && !DROP && !MASKT && QG == 1 && KG == 1 && NW == 8 && KT == 4 && D <= 64), "the pipelined loop has no side inputs");
  constexpr int FRING = 4, VRING = 3;   // fragment reads in flight ahead of their MFMA (K row-major / V transposed)
  using E = Elem<T>;
  using V8 = typename E::V8;
  using C = SwzCfg<D>;
  constexpr int BM = 32 * QG * RG;
  constexpr int TILEB = BN * C::PITCH;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  ACCT_LDS char* smem = (ACCT_LDS char*)smem_raw;   // [2 buffers][K tile | V tile]; reused by the epilogue

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: everything derived from it stays in scalar registers
  const int rg = KG > 1 ? wave % RG : wave, kg = KG > 1 ? wave / RG : 0;
  const int BH = a.B * a.N, n_wg = BH * a.n_tiles;
  int wg = blockIdx.x, slice = 0;                           // kv_split > 1: the grid holds every query tile once per key slice
  if (a.kv_split > 1) split_map(blockIdx.x, BH, a.n_tiles, a.kv_split, a.kv_share, slice, wg);
  int bh, rank;
  wg_map(wg, BH, a.n_tiles, bh, rank);
  const int qt = a.n_tiles - 1 - rank;                      // heaviest (latest) causal tiles first
  const int b = bh / a.N, h = bh % a.N;
  const int q0 = qt * BM;
  const int wq0 = q0 + rg * 32 * QG;                        // first query row of this wave
  const int q_end = min(q0 + BM, a.Sq);                     // one past the last valid row of the block
  const int wq_end = min(wq0 + 32 * QG, a.Sq);

  const T* qp = (const T*)a.q + b * a.q_sb + h * a.q_sh;
  const T* kp = (const T*)a.k + b * a.k_sb + h * a.k_sh;
  const T* vp = (const T*)a.v + b * a.v_sb + h * a.v_sh;

  // ---- visible kv tiles of this block (128-block band; causal and row-prefix clip the top) ----
  const int qb_lo = q0 / 128, qb_hi = (q_end - 1) / 128;
  const int kvb_lo = max(0, qb_lo - a.prev_blk), kvb_hi = min(a.Tc - 1, qb_hi + a.next_blk);
  int j_lo = kvb_lo * 128 / BN, j_hi = min(kvb_hi * 128 + 127, a.Sk - 1) / BN;
  const bool causal = a.mask_kind == kMaskCausal;
  if (causal) j_hi = min(j_hi, (q_end - 1) / BN);
  if (a.row_prefix) j_hi = min(j_hi, (((q_end - 1) / a.row_prefix + 1) * a.row_prefix - 1) / BN);
  const int wqb = wq0 / 128;                                // 128-block of this wave's rows
  BlkClassWindow flwin;                                     // block classes of a dense mask: 64 blocks at a time in scalar registers
  bool flwin_ready = false;
  if (MASKT && a.mask_kind == kMaskDense) {
    // tiles at either end whose 128x128 blocks are wholly masked for every row block of this workgroup are
    // not streamed at all (key padding: the padded tail of every sequence).  With at most 64 blocks in the
    // band, one round trip to memory yields both the trimmed range and the wave's class window.
    const uint8_t* fl = a.blkflags + ((int64_t)(a.mask_sb ? b : 0) * a.Tr) * a.Tc;
    int b_lo = j_lo * BN / 128, b_hi = min((j_hi * BN + BN - 1) / 128, a.Tc - 1);
    const uint8_t* tails = a.blktail ? a.blktail + ((int64_t)(a.mask_sb ? b : 0) * a.Tr) * a.Tc : nullptr;
    if (j_lo <= j_hi && flwin.init_trimmed(fl, 1, a.Tc, qb_lo, qb_hi - qb_lo + 1, min(wqb, qb_hi), b_lo, b_hi, lane, tails)) {
      j_lo = max(j_lo, b_lo * 128 / BN);
      j_hi = min(j_hi, (b_hi * 128 + 127) >> __builtin_ctz(BN));    // (b_hi is -1 when nothing is left)
      flwin_ready = true;
    } else {
      auto dead = [&](int j) {
        for (int kb = j * BN / 128; kb <= min((j * BN + BN - 1) / 128, a.Tc - 1); kb++)
          for (int qb = qb_lo; qb <= qb_hi; qb++)
            if (fl[(int64_t)qb * a.Tc + kb] != kBlkSkip) return false;
        return true;
      };
      trim_dead_tiles(j_lo, j_hi, lane, dead);
    }
  }
  if (a.kv_split > 1) {                                     // this workgroup's slice of the tiles it sees
    const int n = max(j_hi - j_lo + 1, 0), lo = j_lo;
    j_lo = lo + (int)((int64_t)n * slice / a.kv_split);
    j_hi = lo + (int)((int64_t)n * (slice + 1) / a.kv_split) - 1;
  }
  const int wkv_limit = a.row_prefix ? (wq0 / a.row_prefix + 1) * a.row_prefix : 0x7fffffff;   // keys past it are absent

  // ---- the first tile is requested ahead of everything that can be done meanwhile (but see first_tile_late) ----
  TileDma<T, D, BN, NW> kdma, vdma;
  const int cpr = a.hd >> 3;                                // valid 16-byte chunks per row
  kdma.plan(a.k_ss, cpr);
  vdma.plan(a.v_ss, cpr);
  // stage key rows [j BN, (j+1) BN) into an LDS tile (whole tiles by plan; the ragged one's code stands out of the way: 4 to 6 %
  // of a small call at head dim 256, one of 128 1 %)
  auto stage_k = [&](int j, ACCT_LDS char* dst) {
    if (__builtin_expect((j + 1) * BN <= a.Sk, 1)) kdma.issue(kp, a.k_ss, j * BN, dst);
    else tile_dma<T, D, BN, NW>(kp, a.k_ss, j * BN, a.Sk, dst, cpr);         // ragged last tile: clamped rows
  };
  auto stage_v = [&](int j, ACCT_LDS char* dst) {
    if (__builtin_expect((j + 1) * BN <= a.Sk, 1)) vdma.issue(vp, a.v_ss, j * BN, dst);
    else tile_dma<T, D, BN, NW, true>(vp, a.v_ss, j * BN, a.Sk, dst, cpr);   // and zeros
  };
  const bool late = KG <= 2 && !PIPE && D >= 64 && D <= 128 && a.first_late;
  if (j_lo <= j_hi && !late) {
    stage_k(j_lo, smem);
    stage_v(j_lo, smem + TILEB);
  }

  // ---- Q fragments (B operand of K Q^T): lane holds row l32, d = 16t + 8g .. +7 ----
  V8 qf[QG][C::KS];
#pragma unroll
  for (int gq = 0; gq < QG; gq++) {
    const int row = min(wq0 + 32 * gq + l32, a.Sq - 1);     // rows past Sq repeat the last row; never stored
#pragma unroll
    for (int t = 0; t < C::KS; t++) {
      // k-steps (or the upper half of one) past the head dim: zeros there make the products ignore whatever
      // the K tile holds in those slots
      const bool inside = 16 * t + 8 * g < a.hd;
      V8 z;
#pragma unroll
      for (int e = 0; e < 8; e++) z[e] = 0;
      qf[gq][t] = inside ? *reinterpret_cast<const V8*>(qp + (int64_t)row * a.q_ss + 16 * t + 8 * g) : z;
    }
  }

  // ---- per-lane LDS offsets (tile-invariant) ----
  // K fragment of k-step t: row l32, chunk 2t + g.  Chunk c + 8 of a row sits in slot (c ^ swz) ^ 8, so the
  // offsets of the upper half of the head dim are one XOR away from the lower four (wide rows only).
  constexpr int NKOFF = (C::CH >= 16 && C::KS > 4) ? 4 : C::KS;
  int koff_[NKOFF];
#pragma unroll
  for (int t = 0; t < NKOFF; t++) koff_[t] = l32 * C::PITCH + swz_off(2 * t + g, C::swz(l32));
  auto koff = [&](int t) { return t < NKOFF ? koff_[t] : (koff_[t & 3] ^ ((t >> 2) * 128)); };
  const int trow = 4 * g + ((lane & 15) >> 2);              // transposed reads: row within an 8-row group
  const int tchunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  int voff[C::DB];                                          // V^T fragment of d block db
#pragma unroll
  for (int db = 0; db < C::DB; db++) voff[db] = trow * C::PITCH + swz_off(4 * db + tchunk, C::swz(trow)) + 8 * (lane & 1);

  f32x16 o[QG][C::DB];
  float m[QG], lsum[QG];
#pragma unroll
  for (int gq = 0; gq < QG; gq++) {
    // (finite: the first keys a key group or a key slice sees may all be hidden from a row, and -inf - -inf is NaN)
    m[gq] = -1e30f;
    lsum[gq] = 0.f;
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[gq][db][r] = 0.f;
  }

  // Scores stay in raw q.k units (exp2 argument = s * scale*log2e - m * scale*log2e, one FMA) unless a
  // bias is added, in which case they become scale*s + bias first (one mixed-precision FMA per score:
  // the fp16 / bf16 bias is an operand as it is).
  // A key-only bias (row stride 0) that the DMA can stage goes in as the INITIAL value of the score accumulators
  // instead (bias / scale, the MFMAs add q.k): the scores stay in raw units and nothing is spent per score.  The launcher
  // picks 128-key tiles for such a bias and for no other.
  constexpr bool acc_bias = BIAS && KT == 4;
  constexpr bool scaled = BIAS && !acc_bias;                   // scores are turned into scale*s + bias before the softmax
  const bool bias_staged = acc_bias || (scaled && bias_stageable(a));
  const float cmul = scaled ? kLog2e : a.scale_log2e;
  const float madd = scaled ? kMaskFill : a.mask_add_raw;          // the additive -10000 in the units of s
  const float lazy_thr = 8.0f / cmul;                              // 8 octaves, in the units of s
  const int mb = a.mask_sb ? b : 0;
  const uint8_t* maskp = a.mask ? a.mask + (a.mask_kind == kMaskDense ? (int64_t)mb * a.mask_sb * a.mask_es : 0) : nullptr;
  const T* alibip = BIAS ? (const T*)a.alibi + b * a.al_sb + h * a.al_sh : nullptr;
  // (named here and not compared where it is used: with this value among what the softmax lambda captures the compiler
  // allocates the head dim 256 kernel with 758 moves between the two register files instead of 826, and the mask and
  // dropout variants likewise: 32 heads, 3000 x 3000 358 -> 350 us)
  const bool mask_dense = a.mask_kind == kMaskDense;
  const bool alibi_vec = BIAS && (((uintptr_t)a.alibi & 7) | ((a.al_sb | a.al_sh | a.al_sq) & 3)) == 0;

  // bias tiles of this wave's rows are staged through a wave-private LDS region one tile ahead
  // (with 128-key tiles only the key-only form is served: two 256-byte rows per wave)
  constexpr int BIASB = BIAS ? (KT == 4 ? 1024 : QG * 4096) : 0;
  static_assert(KT == 2 || !BIAS || QG == 1, "128-key tiles with a bias: 32 rows per wave");
  ACCT_LDS char* bias_lds = smem + 4 * TILEB + wave * BIASB;
  // (a key-only bias: rows of consecutive tiles alternate between two 256-byte slots of the region, so the next
  // one is requested together with the next K/V tile; a tile bias has one slot and is requested once read)
  auto stage_bias = [&](int jn) {
#pragma unroll
    for (int gq = 0; gq < QG; gq++) {
      if constexpr (acc_bias) bias_row_dma<T>(alibip, jn * BN, a.Sk, bias_lds + (jn & 1) * 256);
      else bias_tile_dma<T>(alibip, a.al_sq, wq0 + 32 * gq, a.Sq, jn * 64, a.Sk, bias_lds + gq * 4096);
    }
  };
  // The staged row of a key-only bias becomes float32 / scale behind its two slots, once per tile and wave, and is the C
  // operand of the first product from there: nothing per score.
  auto convert_bias = [&](int jn) {
    const typename E::V2 v = *reinterpret_cast<const ACCT_LDS typename E::V2*>(bias_lds + (jn & 1) * 256 + lane * 4);
    const f32x2 f = {(float)v[0] * a.inv_scale, (float)v[1] * a.inv_scale};
    *reinterpret_cast<ACCT_LDS f32x2*>(bias_lds + 512 + lane * 8) = f;
  };
  // keep bits of this wave's rows and one tile, staged with the tile's DMA (double buffered)
  using DropStage = DropRowStage<DROP, QG, KT>;
  ACCT_LDS char* drop_lds = smem + 4 * TILEB + NW * BIASB + wave * (2 * DropStage::BYTES);
  // ---- the phases of a tile step: classification, S^T = K Q^T, online softmax, O^T += V^T P^T ----
  const uint8_t* flrow = (MASKT && a.mask_kind == kMaskDense) ? a.blkflags + ((int64_t)mb * a.Tr + wqb) * a.Tc : nullptr;
  if (!flwin_ready && j_lo <= j_hi)
    flwin.init(flrow, 1, j_lo * BN / 128, min((j_hi * BN + BN - 1) / 128, a.Tc - 1), lane, (flrow && a.blktail) ? a.blktail + (flrow - a.blkflags) : nullptr);
  enum : uint32_t { kAct = 1u, kApply = 2u, kDiag = 4u, kTailShift = 8u };   // bits 8..15: key tail of the tile's block (0: none)
  // what this wave does with tile j (tiles must be asked for in ascending order)
  auto classify = [&](int j) -> uint32_t {
    const int kv0 = j * BN + kg * WN, kvb = kv0 / 128;
    const uint32_t fl_cur = flwin.get(kvb, lane);
    bool act = (kvb - a.next_blk <= wqb) && (wqb <= kvb + a.prev_blk) && (wq0 < a.Sq);
    if (causal) act = act && (kv0 <= wq_end - 1);
    act = act && (kv0 < wkv_limit);
    if (KG > 1) act = act && (kv0 < a.Sk);
    bool apply_mask = false;
    bool diag = causal;                                     // keys after the query are hidden, by index compare
    uint32_t tail = 0;
    if (MASKT && a.mask_kind == kMaskDense && act) {
      act = fl_cur != kBlkSkip;
      apply_mask = fl_cur == kBlkApply;
      if (fl_cur == kBlkTriu) { diag = true; act = kv0 <= wq_end - 1; }
      if (apply_mask && (tail = flwin.tail(kvb)) != 0) {
        // every row of the block hides exactly the keys from its tail-th on: an index compare, no mask loads
        apply_mask = false;
        act = kv0 < kvb * 128 + (int)tail;
      }
    } else if (MASKT && a.mask_kind == kMaskTile) {
      apply_mask = wqb == kvb;
    }
    return (act ? kAct : 0u) | (apply_mask ? kApply : 0u) | (diag ? kDiag : 0u) | (tail << kTailShift);
  };
  // S^T = K Q^T : s[gq][c] is the 32(kv) x 32(q) tile of kv chunk c
  auto gemm_s = [&](const ACCT_LDS char* kbuf, int j, f32x16 (&s)[QG][KTW]) {
    if (BIAS && acc_bias) {
      // element (c, r) belongs to key 32 c + 8 (r/4) + 4 g + r%4 of the tile, whatever the lane's row
#pragma unroll
      for (int gq = 0; gq < QG; gq++)
#pragma unroll
        for (int c = 0; c < KTW; c++)
#pragma unroll
          for (int r4 = 0; r4 < 4; r4++) {
            const f32x4 bv = *reinterpret_cast<const ACCT_LDS f32x4*>(bias_lds + 512 + (32 * (kg * KTW + c) + 8 * r4 + 4 * g) * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) s[gq][c][4 * r4 + e] = bv[e];
          }
    } else {
#pragma unroll
      for (int gq = 0; gq < QG; gq++)
#pragma unroll
        for (int c = 0; c < KTW; c++)
#pragma unroll
          for (int r = 0; r < 16; r++) s[gq][c][r] = 0.f;
    }
    // K fragments travel through a ring of FRING register sets: FRING reads are in flight ahead of the
    // MFMA that consumes the oldest one, so that a wave covers the LDS latency (well over one MFMA) by
    // itself.  The scheduling barriers keep the compiler from folding the ring back into read-wait-MFMA.
    constexpr int NF = KTW * C::KS;
    constexpr int RING = FRING < NF ? FRING : NF;
    V8 ring[RING];
    auto kread = [&](int i) { return lds_read_frag<T>(kbuf + koff(i % C::KS) + (i / C::KS) * 32 * C::PITCH); };
#pragma unroll
    for (int i = 0; i < RING; i++) ring[i] = kread(i);
#pragma unroll
    for (int i = 0; i < NF; i++) {
      const int c = i / C::KS, t = i % C::KS;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int gq = 0; gq < QG; gq++) s[gq][c] = E::mfma(ring[i % RING], qf[gq][t], s[gq][c]);
      if (i + RING < NF)
        ring[i % RING] = kread(i + RING);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // O^T += V^T P^T, the transposed V fragments through a ring as well
  auto gemm_pv = [&](const ACCT_LDS char* vbuf, const V8 (&pf)[QG][KTW][2]) {
    constexpr int NT = 2 * KTW * C::DB;
    constexpr int RING = VRING < NT ? VRING : NT;
    auto tread = [&](int i) {
      const int db = i % C::DB, ch = i / C::DB;               // ch = 2 c + hh: rows 16 ch .. of the tile
      const ACCT_LDS char* vaddr = vbuf + voff[db] + 16 * ch * C::PITCH;
      return join_tr<T>(lds_read_tr(vaddr), lds_read_tr(vaddr + C::tr_hi(db)));
    };
    V8 ring[RING];
#pragma unroll
    for (int i = 0; i < RING; i++) ring[i] = tread(i);
#pragma unroll
    for (int i = 0; i < NT; i++) {
      const int db = i % C::DB, ch = i / C::DB;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int gq = 0; gq < QG; gq++) o[gq][db] = E::mfma(ring[i % RING], pf[gq][ch >> 1][ch & 1], o[gq][db]);
      if (i + RING < NT) ring[i % RING] = tread(i + RING);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // online softmax of the scores of tile j -> P^T fragments; `buf` = parity of the tile's staging buffers
  auto softmax = [&](int j, int buf, uint32_t info, f32x16 (&s)[QG][KTW], V8 (&pf)[QG][KTW][2]) {
    const int kv0 = j * BN + kg * WN;
    const bool apply_mask = MASKT && (info & kApply), diag = info & kDiag;
    const int tail = MASKT ? (int)((info >> kTailShift) & 0xffu) : 0;
    const int last_key = tail ? min(a.Sk, kv0 / 128 * 128 + tail) - 1 : a.Sk - 1;     // last key that exists and is not behind a key tail
    // element (gq, c, r): q = wq0 + 32 gq + l32 ; kv = kv0 + 32 c + 8 (r/4) + 4 g + r%4
    const bool edge = apply_mask || (diag && (kv0 + WN - 1 > wq0)) || (kv0 + WN - 1 > last_key);
#pragma unroll
    for (int gq = 0; gq < QG; gq++) {
      const int qrow = wq0 + 32 * gq + l32;
      const int qrow_c = min(qrow, a.Sq - 1);            // clamped for side-input addressing
      if (BIAS && !acc_bias) {
        if (bias_staged) {
          constexpr int KB = KT == 2 ? KTW : 1;                // (this path is that of the 64-key tiles)
          typename E::V4 bv[KB][4];
#pragma unroll
          for (int c = 0; c < KB; c++)
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) bv[c][r4] = bias_tile_read<T>(bias_lds + gq * 4096, l32, 4 * (kg * KTW + c) + r4, g);
          if (gq == QG - 1) {
            // the tile is in registers: its LDS region can take the next tile, which has the rest of
            // this step to land (the end-of-step wait covers it)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (j < j_hi) stage_bias(j + 1);
          }
#pragma unroll
          for (int c = 0; c < KB; c++)
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++)
#pragma unroll
              for (int e = 0; e < 4; e++)
                s[gq][c][4 * r4 + e] = __builtin_fmaf(s[gq][c][4 * r4 + e], a.scale, (float)bv[c][r4][e]);
        } else {
#pragma unroll
          for (int c = 0; c < KTW; c++)
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) {
              const int kv = kv0 + 32 * c + 8 * r4 + 4 * g;
              float bias[4];
              load_bias4<T>(alibip + (int64_t)qrow_c * a.al_sq, kv, a.Sk, alibi_vec, bias);
#pragma unroll
              for (int e = 0; e < 4; e++)
                s[gq][c][4 * r4 + e] = __builtin_fmaf(s[gq][c][4 * r4 + e], a.scale, bias[e]);
            }
        }
      }
      if (edge) {
        if (apply_mask) {
#pragma unroll
          for (int c = 0; c < KTW; c++)
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) {
              const int kv = kv0 + 32 * c + 8 * r4 + 4 * g;
              uint32_t mbits;
              if (mask_dense) mbits = load_mask4(maskp + (int64_t)qrow_c * a.Sk * a.mask_es, kv, a.Sk, a.mask_es);
              else mbits = load_mask4(maskp + (qrow_c & 127) * 128 * a.mask_es, kv & 127, 128, a.mask_es);
#pragma unroll
              for (int e = 0; e < 4; e++)
                if ((mbits >> (8 * e)) & 0xffu) s[gq][c][4 * r4 + e] += madd;
            }
        }
        {
          // Keys after the query (causal diagonal) and keys past Sk are removed outright: with the additive
          // mask their probability underflows to exactly 0 as well (the diagonal key is always visible), so
          // the result is the same bit for bit at a third of the vector instructions.
          int vis = last_key - kv0 - 4 * g;                  // last visible key, relative to this lane's first
          if (diag) vis = min(vis, qrow - kv0 - 4 * g);
          // (compare and select through VCC: see select_if_gt)
          const float ninf = -INFINITY;
#pragma unroll
          for (int c = 0; c < KTW; c++) {
            const int visc = vis - 32 * c;
#pragma unroll
            for (int r = 0; r < 16; r++) s[gq][c][r] = select_if_gt(s[gq][c][r], 8 * (r >> 2) + (r & 3), visc, ninf);
          }
        }
      }
      // ---- online softmax for query row qrow ----
      float mx = s[gq][0][0];
#pragma unroll
      for (int c = 0; c < KTW; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[gq][c][r]);
      mx = pair_max(mx);
      // Lazy running max: it only moves when a score beats it by more than 2^8 in probability
      // terms.  Until then P = exp2(s - m) may reach 256 instead of 1 (harmless in fp16/bf16 and in
      // the fp32 sums; O = acc / l and LSE = m + ln l are unchanged), and the O rescale below is
      // skipped for almost every tile after the first.
      const bool grow = mx > m[gq] + lazy_thr;
      const float m_new = grow ? mx : m[gq];
      const float alpha = grow ? fast_exp2((m[gq] - m_new) * cmul) : 1.0f;
      const float mc = m_new * cmul;
      m[gq] = m_new;
      float rs = 0.f;
      float p[KTW][16];
#pragma unroll
      for (int c = 0; c < KTW; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          p[c][r] = fast_exp2(__builtin_fmaf(s[gq][c][r], cmul, -mc));
          rs += p[c][r];
        }
      lsum[gq] = lsum[gq] * alpha + rs;                  // row sum BEFORE dropout
      if (DROP) {
        // keep bits of this row and tile: word c covers keys kv0 + 32c .. +31
#pragma unroll
        for (int c = 0; c < KTW; c++) {
          const uint32_t w = DropStage::word(drop_lds + buf * DropStage::BYTES, 32 * gq + l32, kg * KTW + c) >> (4 * g);
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int32_t sel = __builtin_amdgcn_sbfe((int)w, 8 * (r >> 2) + (r & 3), 1);   // keep ? ~0 : 0
            p[c][r] = __uint_as_float(__float_as_uint(p[c][r]) & (uint32_t)sel);        // (1 / keep_prob: once, on O)
          }
        }
      }
#pragma unroll
      for (int c = 0; c < KTW; c++)
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
          typename E::V2 t0 = E::cvt2(p[c][8 * hh + 0], p[c][8 * hh + 1]);
          typename E::V2 t1 = E::cvt2(p[c][8 * hh + 2], p[c][8 * hh + 3]);
          typename E::V2 t2 = E::cvt2(p[c][8 * hh + 4], p[c][8 * hh + 5]);
          typename E::V2 t3 = E::cvt2(p[c][8 * hh + 6], p[c][8 * hh + 7]);
          V8 pv = {t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
          pf[gq][c][hh] = pv;
        }
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int db = 0; db < C::DB; db++)
#pragma unroll
          for (int r = 0; r < 16; r++) o[gq][db][r] *= alpha;
      }
    }
  };

  if constexpr (PIPE) {
    // ---- tile loop, pipelined: step j issues O^T += V(j-1)^T P(j-1)^T and S(j+1)^T = K(j+1) Q^T with the softmax of tile j
    // between their MFMAs.  The eight waves start a step together, so in the plain loop below the two of a SIMD are in their
    // matrix phases at the same time and then both in the softmax.  Needs two tiles of scores and the packed P in registers:
    // up to head dim 64 (with 64-key tiles head dims 80 and 128 lose 3 % to the plain loop).  For long walks: pipelined_pays,
    // which has both sides' times ----
    // this wave's own tiles
    const int key_end = min(min(causal ? wq_end : a.Sk, wkv_limit), a.Sk) - kg * WN;
    const int w_lo = max(j_lo, max(0, wqb - a.prev_blk) * 128 / BN);
    const int w_hi = wq0 < a.Sq && key_end > 0 ? min(min(j_hi, (min(a.Tc - 1, wqb + a.next_blk) * 128 + 127) / BN), (key_end - 1) / BN) : -1;
    constexpr int NPV = 2 * KTW * C::DB, NQK = KTW * C::KS, NM = NPV + NQK, NE = 16 * KTW;
    // buffers of step j: it reads those of the other parity and fills its own
    int par = 0;                                             // byte offset of step j's own buffers
    const T *kfill = kp + (int64_t)(j_lo + 2) * BN * a.k_ss, *vfill = vp + (int64_t)j_lo * BN * a.v_ss;   // what step j requests
    const int64_t kstep = BN * a.k_ss, vstep = BN * a.v_ss;
    auto fill = [&](int j) {
      if (j + 2 <= j_hi) {
        if ((j + 3) * BN <= a.Sk) kdma.issue(kfill, a.k_ss, 0, smem + par);
        else tile_dma<T, D, BN, NW>(kp, a.k_ss, (j + 2) * BN, a.Sk, smem + par, cpr);     // ragged last tile: clamped rows
      }
      if (j > j_lo && j <= j_hi) {                           // (that of the first tile is under way)
        if (__builtin_expect((j + 1) * BN <= a.Sk, 1)) vdma.issue(vfill, a.v_ss, 0, smem + par + TILEB);
        else tile_dma<T, D, BN, NW, true>(vp, a.v_ss, j * BN, a.Sk, smem + par + TILEB, cpr);
      }
      kfill += kstep;
      vfill += vstep;
    };
    auto publish = [&] {
      par ^= 2 * TILEB;
      dma_wait();
      __syncthreads();
    };
    // (a tile before the wave's last: all of its keys exist, and under the causal mask they come before the wave's first row)
    auto fused = [&](int j, f32x16 (&s)[1][KTW], f32x16 (&sn)[1][KTW], V8 (&pf)[1][KTW][2]) {
      const ACCT_LDS char* kbuf = smem + (par ^ (2 * TILEB));
      const ACCT_LDS char* vbuf = kbuf + TILEB;
#pragma unroll
      for (int c = 0; c < KTW; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) sn[0][c][r] = 0.f;
      constexpr int RING = 4;
      auto fread = [&](int i) {
        if (i < NPV) {
          const ACCT_LDS char* vaddr = vbuf + voff[i % C::DB] + 16 * (i / C::DB) * C::PITCH;
          return join_tr<T>(lds_read_tr(vaddr), lds_read_tr(vaddr + C::tr_hi(i % C::DB)));
        }
        return lds_read_frag<T>(kbuf + koff((i - NPV) % C::KS) + ((i - NPV) / C::KS) * 32 * C::PITCH);
      };
      V8 ring[RING];
      uint32_t pn[NE / 2];
#pragma unroll
      for (int i = 0; i < RING; i++) ring[i] = fread(i);
      // vector work in the order it depends on itself, dealt out over the MFMAs by its cycles
      constexpr int CM = 2, CS = 24, CE = 7, CT = NE / 2 * CM + CS + NE * CE;
      float mx = s[0][0][0], mx1 = s[0][0][2], mc = 0.f, alpha = 1.f, rs = 0.f, p[2];
#pragma unroll
      for (int i = 0; i < NM; i++) {
        __builtin_amdgcn_sched_barrier(0);
        if (i < NPV) o[0][i % C::DB] = E::mfma(ring[i % RING], pf[0][(i / C::DB) >> 1][(i / C::DB) & 1], o[0][i % C::DB]);
        else sn[0][(i - NPV) / C::KS] = E::mfma(ring[i % RING], qf[0][(i - NPV) % C::KS], sn[0][(i - NPV) / C::KS]);
        if (i + RING < NM) ring[i % RING] = fread(i + RING);
        if (i == 1) fill(j);                                 // (behind the first fragment reads, whose latency it covers)
#pragma unroll
        for (int k = 0; k < NE / 2; k++)
          if (k * CM * NM / CT == i) {
            float& m2 = k & 1 ? mx1 : mx;                    // (two chains: a dependent maximum waits 8 cycles, issues in 4)
            m2 = fmaxf(fmaxf(m2, s[0][k / 8][2 * (k & 7)]), s[0][k / 8][2 * (k & 7) + 1]);
          }
        if (NE / 2 * CM * NM / CT == i) {
          mx = pair_max(fmaxf(mx, mx1));
          const bool grow = mx > m[0] + lazy_thr;
          const float m_new = grow ? mx : m[0];
          alpha = grow ? fast_exp2((m[0] - m_new) * cmul) : 1.0f;
          mc = m_new * cmul;
          m[0] = m_new;
        }
#pragma unroll
        for (int e = 0; e < NE; e++)
          if ((NE / 2 * CM + CS + e * CE) * NM / CT == i) {
            p[e & 1] = fast_exp2(__builtin_fmaf(s[0][e / 16][e & 15], cmul, -mc));
            rs += p[e & 1];
            if (e & 1) {
              // (pinned here: the compiler would move all of it behind the barrier, to where the next step uses it)
              pn[e / 2] = __builtin_bit_cast(uint32_t, E::cvt2(p[0], p[1]));
              asm volatile("" : "+v"(pn[e / 2]), "+v"(rs));
            }
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      lsum[0] = lsum[0] * alpha + rs;
#pragma unroll
      for (int c = 0; c < KTW; c++)
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
          const u32x4 t = {pn[8 * c + 4 * hh], pn[8 * c + 4 * hh + 1], pn[8 * c + 4 * hh + 2], pn[8 * c + 4 * hh + 3]};
          pf[0][c][hh] = __builtin_bit_cast(V8, t);
        }
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int db = 0; db < C::DB; db++)
#pragma unroll
          for (int r = 0; r < 16; r++) o[0][db][r] *= alpha;
      }
    };
    f32x16 s0[1][KTW], s1[1][KTW];
    V8 pf[1][KTW][2];
    auto step = [&](int j) {
      const ACCT_LDS char* buf = smem + (par ^ (2 * TILEB)) + kg * (WN * C::PITCH);
      fill(j);
      if (j > w_lo && j - 1 <= w_hi) gemm_pv(buf + TILEB, pf);
      if (j >= w_lo && j <= w_hi) softmax(j, 0, kAct | (causal ? kDiag : 0u), s0, pf);
      if (j + 1 >= w_lo && j + 1 <= w_hi) gemm_s(buf, j + 1, s0);
      publish();
    };
    if (j_lo <= j_hi) {
      if (j_lo < j_hi) stage_k(j_lo + 1, smem + 2 * TILEB);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (j_lo == w_lo && j_lo <= w_hi) gemm_s(smem + kg * (WN * C::PITCH), j_lo, s0);
      __syncthreads();
      int j = j_lo;
      for (; j <= min(w_lo, j_hi + 1); j++) step(j);
      for (; j + 1 < w_hi; j += 2) {
        fused(j, s0, s1, pf);
        publish();
        fused(j + 1, s1, s0, pf);
        publish();
      }
      for (; j <= j_hi + 1; j++) step(j);
    }
  } else if (j_lo <= j_hi) {
    if (late) {
      stage_k(j_lo, smem);
      stage_v(j_lo, smem + TILEB);
    }
    if (BIAS && bias_staged && wq0 < a.Sq) stage_bias(j_lo);
    DropStage::issue(a, bh, wq0, j_lo, lane, drop_lds);
    // A full wait the compiler can see: every load issued so far (Q fragments included) is complete, so
    // it places no vmcnt wait inside the loop -- such a wait would also stall on the next tile's DMA.
    __builtin_amdgcn_s_waitcnt(0);
    if (acc_bias) convert_bias(j_lo);
    __syncthreads();
    for (int j = j_lo; j <= j_hi; j++) {
      const int buf = (j - j_lo) & 1;
      ACCT_LDS char* kbuf = smem + buf * 2 * TILEB;
      ACCT_LDS char* vbuf = kbuf + TILEB;
      if (j < j_hi) {                                       // next tile streams into the other buffer meanwhile
        ACCT_LDS char* nb = smem + (buf ^ 1) * 2 * TILEB;
        stage_k(j + 1, nb);
        stage_v(j + 1, nb + TILEB);
        DropStage::issue(a, bh, wq0, j + 1, lane, drop_lds + (buf ^ 1) * DropStage::BYTES);
        if (BIAS && acc_bias && wq0 < a.Sq) stage_bias(j + 1);
      }
      const uint32_t info = classify(j);
      if (info & kAct) {
        f32x16 s[QG][KTW];
        V8 pf[QG][KTW][2];
        gemm_s(kbuf + kg * (WN * C::PITCH), j, s);
        softmax(j, buf, info, s, pf);
        gemm_pv(vbuf + kg * (WN * C::PITCH), pf);
      } else if (BIAS && bias_staged && !acc_bias && j < j_hi && wq0 < a.Sq) {
        stage_bias(j + 1);                                  // nothing to read in this step: the region is free
      }
      dma_wait();
      if (acc_bias && j < j_hi) convert_bias(j + 1);
      __syncthreads();
    }
  }

  // ---- key groups: each finishes its share of the columns from the sums of all.  (One group merging and storing all of
  // them while the others idled: 3900 cycles from the last tile on, of a workgroup that walked four tiles in 8000, D64, kg 4;
  // shared 2400.)  Not in a launch of several rounds at head dims up to 64: there the others are better gone, as three waves
  // fit a SIMD and the next workgroup starts beside the first group's merge.  Forward, shared / alone (us): 1024 heads,
  // 300 x 77, key padding, D40 71.6 / 65.2, D64 73.7 / 66.9; dropout 58.9 / 53.2, 66.9 / 59.2; 384 heads, 300 x 300 padded 35.6 / 32.9,
  // 39.7 / 36.9; 24 heads, 3000 x 500 28.9 / 27.8, 29.1 / 27.5; without side inputs level.  The sums and their order are the same. ----
  bool merged = false;
  if constexpr (fwd_merge_alone<D, KG>()) if (a.merge_alone) {
    merged = true;
    ACCT_LDS char* slot = smem + RG * 32 * (C::DB * 64 + 16) + rg * (C::DB * 4096 + 512) + lane * 16;
    ACCT_LDS char* stat = slot + C::DB * 4096 - lane * 8;
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < 4 * C::DB; i++) {
        const f32x4 v = {o[0][i / 4][4 * (i % 4)], o[0][i / 4][4 * (i % 4) + 1], o[0][i / 4][4 * (i % 4) + 2], o[0][i / 4][4 * (i % 4) + 3]};
        *reinterpret_cast<ACCT_LDS f32x4*>(slot + i * 1024) = v;
      }
      *reinterpret_cast<ACCT_LDS f32x2*>(stat) = f32x2{m[0], lsum[0]};
    }
    __syncthreads();
    if (kg > 0) return;
    const f32x2 ml = *reinterpret_cast<const ACCT_LDS f32x2*>(stat);
    const float mm = fmaxf(m[0], ml[0]), w0 = fast_exp2((m[0] - mm) * cmul), w1 = fast_exp2((ml[0] - mm) * cmul);
    m[0] = mm;
    lsum[0] = __builtin_fmaf(ml[1], w1, lsum[0] * w0);
#pragma unroll
    for (int i = 0; i < 4 * C::DB; i++) {
      const f32x4 v = *reinterpret_cast<const ACCT_LDS f32x4*>(slot + i * 1024);
#pragma unroll
      for (int e = 0; e < 4; e++) o[0][i / 4][4 * (i % 4) + e] = __builtin_fmaf(v[e], w1, o[0][i / 4][4 * (i % 4) + e] * w0);
    }
  }
  if constexpr (KG > 1) if (!merged) {
    constexpr int PC = fwd_merge_pieces<D, KG>();
    static_assert(PC * KG == 4 * C::DB, "every key group finishes the same number of pieces");
    // pieces of key group `own` that key group `from` holds
    auto slot = [&](int own, int from) {
      return smem + ((rg * KG + own) * (KG - 1) + from - (from > own ? 1 : 0)) * (PC * 1024) + lane * 16;
    };
    ACCT_LDS char* stats = smem + fwd_merge_stats<D, NW, KG>() + rg * (KG * 512) + lane * 8;
    auto piece = [&](int i) -> f32x4 {
      return {o[0][i / 4][4 * (i % 4)], o[0][i / 4][4 * (i % 4) + 1], o[0][i / 4][4 * (i % 4) + 2], o[0][i / 4][4 * (i % 4) + 3]};
    };
#pragma unroll
    for (int k = 0; k < KG; k++)
      if (k != kg) {
#pragma unroll
        for (int i = 0; i < PC; i++) *reinterpret_cast<ACCT_LDS f32x4*>(slot(k, kg) + i * 1024) = piece(k * PC + i);
      }
    const f32x2 mine = {m[0], lsum[0]};
    *reinterpret_cast<ACCT_LDS f32x2*>(stats + kg * 512) = mine;
    __syncthreads();
    f32x2 ml[KG];
    float w[KG], mm = -1e30f, l = 0.f;
#pragma unroll
    for (int k = 0; k < KG; k++) {
      ml[k] = *reinterpret_cast<const ACCT_LDS f32x2*>(stats + k * 512);
      mm = fmaxf(mm, ml[k][0]);
    }
#pragma unroll
    for (int k = 0; k < KG; k++) {
      w[k] = fast_exp2((ml[k][0] - mm) * cmul);
      l = k == 0 ? ml[0][1] * w[0] : __builtin_fmaf(ml[k][1], w[k], l);
    }
    l = pair_sum(l);
    f32x4 acc[PC];
#pragma unroll
    for (int own = 0; own < KG; own++)
      if (own == kg) {
#pragma unroll
        for (int i = 0; i < PC; i++)
#pragma unroll
          for (int k = 0; k < KG; k++) {                     // (in the order of the keys, whoever adds)
            const f32x4 v = k == own ? piece(own * PC + i) : *reinterpret_cast<const ACCT_LDS f32x4*>(slot(own, k) + i * 1024);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][e] = k == 0 ? v[e] * w[0] : __builtin_fmaf(v[e], w[k], acc[i][e]);
          }
      }
    if (wq0 >= a.Sq) return;
    if (a.kv_split > 1) {                                    // sums and statistics of a key slice (as below)
      const int64_t idx = ((int64_t)slice * n_wg + wg) * RG + rg, n_idx = (int64_t)a.kv_split * n_wg * RG;
      float* part = a.fwd_part + idx * (C::DB * 1024) + kg * (PC * 256) + lane * 4;
#pragma unroll
      for (int i = 0; i < PC; i++) *reinterpret_cast<f32x4*>(part + i * 256) = acc[i];
      const f32x2 msl = {mm, l};
      if (kg == 0 && g == 0) *reinterpret_cast<f32x2*>(a.fwd_part + n_idx * (C::DB * 1024) + (idx * 32 + l32) * 2) = msl;
      return;
    }
    const int row = wq0 + l32, nch = a.hd >> 3;
    const float inv = l > 0.f ? (DROP ? a.inv_keep : 1.0f) / l : 0.f;
    if (row >= a.Sq) return;
    if (kg == 0 && g == 0) a.lse[(int64_t)bh * a.Sq + row] = l > 0.f ? mm * (scaled ? 1.0f : a.scale) + __logf(l) : -INFINITY;
    T* orow = (T*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)row * a.o_ss;
    // lanes l and l + 32 hold half a 16-byte chunk of two pieces each: they exchange halves and store one whole chunk each
#pragma unroll
    for (int i = 0; i < PC; i += 2) {
      uint32_t t[2][2];
#pragma unroll
      for (int x = 0; x < 2 && i + x < PC; x++) {
        t[x][0] = __builtin_bit_cast(uint32_t, E::cvt2(acc[i + x][0] * inv, acc[i + x][1] * inv));
        t[x][1] = __builtin_bit_cast(uint32_t, E::cvt2(acc[i + x][2] * inv, acc[i + x][3] * inv));
      }
      if (i + 1 < PC) {
        const u32x2 lo = __builtin_amdgcn_permlane32_swap(t[0][0], t[1][0], false, false), hi = __builtin_amdgcn_permlane32_swap(t[0][1], t[1][1], false, false);
        const u32x4 v = {lo[0], hi[0], lo[1], hi[1]};
        const int ch = kg * PC + i + g;
        if (ch < nch) *reinterpret_cast<u32x4*>(orow + ch * 8) = v;
      } else {
        const u32x2 v = {t[0][0], t[0][1]};
        const int ch = kg * PC + i;
        if (ch < nch) *reinterpret_cast<u32x2*>(orow + ch * 8 + 4 * g) = v;
      }
    }
    return;
  }
  // ---- key slices: sums and statistics go to the workspace, fa_fwd_combine_kernel adds the slices up ----
  if (a.kv_split > 1) {
    if (wq0 >= a.Sq) return;
    const int64_t idx = ((int64_t)slice * n_wg + wg) * RG + rg, n_idx = (int64_t)a.kv_split * n_wg * RG;
#pragma unroll
    for (int gq = 0; gq < QG; gq++) {
      float* part = a.fwd_part + (idx * QG + gq) * (C::DB * 1024) + lane * 4;
#pragma unroll
      for (int db = 0; db < C::DB; db++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
          const f32x4 v = {o[gq][db][4 * r4], o[gq][db][4 * r4 + 1], o[gq][db][4 * r4 + 2], o[gq][db][4 * r4 + 3]};
          *reinterpret_cast<f32x4*>(part + (4 * db + r4) * 256) = v;
        }
      const float l = pair_sum(lsum[gq]);
      const f32x2 ml = {m[gq], l};
      if (g == 0) *reinterpret_cast<f32x2*>(a.fwd_part + n_idx * QG * (C::DB * 1024) + ((idx * QG + gq) * 32 + l32) * 2) = ml;
    }
    return;
  }

  // ---- epilogue: O = O^T / l, LSE = m + ln l.  Each wave transposes its rows through its own
  // LDS region (pitch 2D+16 keeps the 8-byte writes of 16 rows on distinct banks) so that the
  // global stores are whole rows. ----
  T* op = (T*)a.o + b * a.o_sb + h * a.o_sh;
  const float mnat = scaled ? 1.0f : a.scale;
  constexpr int OPITCH = C::DB * 64 + 16;
  ACCT_LDS char* obuf = smem + rg * (32 * OPITCH);
#pragma unroll
  for (int gq = 0; gq < QG; gq++) {
    const int row = wq0 + 32 * gq + l32;
    const float l = pair_sum(lsum[gq]);
    const float inv = l > 0.f ? (DROP ? a.inv_keep : 1.0f) / l : 0.f;
    if (row < a.Sq && g == 0) a.lse[(int64_t)bh * a.Sq + row] = l > 0.f ? m[gq] * mnat + __logf(l) : -INFINITY;
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
      for (int r4 = 0; r4 < 4; r4++) {
        typename E::V2 t0 = E::cvt2(o[gq][db][4 * r4 + 0] * inv, o[gq][db][4 * r4 + 1] * inv);
        typename E::V2 t1 = E::cvt2(o[gq][db][4 * r4 + 2] * inv, o[gq][db][4 * r4 + 3] * inv);
        typename E::V4 ov = {t0[0], t0[1], t1[0], t1[1]};
        *reinterpret_cast<ACCT_LDS typename E::V4*>(obuf + l32 * OPITCH + (32 * db + 8 * r4 + 4 * g) * 2) = ov;
      }
    // read back row-contiguous: 16-byte chunk ch of row r
    const int nch = a.hd >> 3;                       // valid 16-byte chunks per row
    const uint32_t nch_inv = recip16(nch);
#pragma unroll
    for (int i = 0; i < (32 * C::CPR + 63) / 64; i++) {
      const int idx = lane + 64 * i;
      const int r = div_small(idx, nch_inv), ch = idx - r * nch;
      const int grow = wq0 + 32 * gq + r;
      if (idx < 32 * nch && grow < a.Sq) {
        const u32x4 v = *reinterpret_cast<const ACCT_LDS u32x4*>(obuf + r * OPITCH + ch * 16);
        *reinterpret_cast<u32x4*>(op + (int64_t)grow * a.o_ss + ch * 8) = v;
      }
    }
  }
}


// The variant that knows mask tensors but neither a bias nor dropout carries a second body: a workgroup whose
// rows see nothing but the causal pattern in a dense mask (block classes: clean before the diagonal, the
// causal diagonal, skipped after it) runs the code of the variant without side inputs, by index compare.
// A causal mask given as a tensor then costs one look at the class table per workgroup.
template <typename T, int D, int QG, int NW, bool BIAS, bool DROP, bool MASKT, int KT = 2, int KG = 1, bool PIPE = false>
__global__ void __launch_bounds__(64 * NW) fa_fwd_kernel(const FaArgs a) {
  if constexpr (MASKT && (!BIAS || KT == 4) && !DROP) {
    if (BIAS && a.mask_kind != kMaskDense && a.mask_kind != kMaskTile) {
      fa_fwd_body<T, D, QG, NW, BIAS, false, false, KT, KG>(a);
      return;
    }
    if (a.mask_kind == kMaskDense) {
      constexpr int BM = 32 * QG * NW / KG;
      const int BH = a.B * a.N;
      int wg = blockIdx.x, slice;
      if (a.kv_split > 1) split_map(blockIdx.x, BH, a.n_tiles, a.kv_split, a.kv_share, slice, wg);
      int bh, rank;
      wg_map(wg, BH, a.n_tiles, bh, rank);
      const int q0 = (a.n_tiles - 1 - rank) * BM, q_end = min(q0 + BM, a.Sq);
      const int qb_lo = q0 / 128, qb_hi = (q_end - 1) / 128;
      const int kvb_lo = max(0, qb_lo - a.prev_blk), kvb_hi = min(a.Tc - 1, qb_hi + a.next_blk);
      const uint8_t* fl = a.blkflags + ((int64_t)(a.mask_sb ? bh / a.N : 0) * a.Tr) * a.Tc;
      if (dense_lines_are_causal(fl, 1, a.Tc, qb_lo, qb_hi - qb_lo + 1, kvb_lo, kvb_hi, false, a, threadIdx.x & 63)) {
        FaArgs c = a;
        c.mask_kind = kMaskCausal;
        fa_fwd_body<T, D, QG, NW, BIAS, false, false, KT, KG, PIPE>(c);
        return;
      }
    }
  }
  fa_fwd_body<T, D, QG, NW, BIAS, DROP, MASKT, KT, KG, PIPE && !MASKT>(a);
}

// Second half of a forward launch whose key range was cut into a.kv_split slices: O = sum_s w_s O_s / sum_s w_s l_s
// with w_s = exp2((m_s - max m) cmul), LSE from the same sums.  One workgroup per 32 query rows and 8 output columns
// (the 1 KB a wave of the first half stored with one instruction), so that a single head's rows still spread over
// the chip; its four waves take every fourth slice, eight loads in flight, and meet in LDS.
template <typename T>
__global__ void __launch_bounds__(256) fa_fwd_combine_kernel(const FaArgs a, int rgs, int dbs, float cmul, float mnat, float omul) {
  __shared__ float red[3][6][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, g = lane >> 5;
  const int BH = a.B * a.N, n_wg = BH * a.n_tiles;
  const int dr = blockIdx.x % (4 * dbs), idx0 = blockIdx.x / (4 * dbs);     // dr = 4 db + r4
  const int rg = idx0 % rgs;
  int bh, rank;
  wg_map(idx0 / rgs, BH, a.n_tiles, bh, rank);
  const int wq0 = ((a.n_tiles - 1 - rank) * rgs + rg) * 32, row = wq0 + l32;
  if (wq0 >= a.Sq) return;
  const int64_t step = (int64_t)n_wg * rgs;
  const float* part = a.fwd_part + (int64_t)idx0 * (dbs * 1024) + dr * 256 + lane * 4;
  const float* stat = a.fwd_part + a.kv_split * step * (dbs * 1024) + ((int64_t)idx0 * 32 + l32) * 2;
  float m = -1e30f, l = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  constexpr int U = 8;
  for (int s0 = wave; s0 < a.kv_split; s0 += 4 * U) {
    f32x4 v[U];
    f32x2 ml[U];
    float mb = m;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int s = min(s0 + 4 * u, a.kv_split - 1);                        // (a repeated slice is left out below)
      v[u] = *reinterpret_cast<const f32x4*>(part + s * step * (dbs * 1024));
      ml[u] = *reinterpret_cast<const f32x2*>(stat + s * step * 64);
    }
#pragma unroll
    for (int u = 0; u < U; u++) mb = fmaxf(mb, ml[u][0]);
    const float al = fast_exp2((m - mb) * cmul);
    m = mb;
    l *= al;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] *= al;
    // (eight whole slices need no test: 6.3 us for 256 queries x 131072 keys, 7.3 with it.  Fewer: selects on values that are
    // loaded in any case -- a branch around each slice serialised the loads, 12.2 us, and a weight of 0 alone would turn an
    // infinity of V into NaN)
    auto add = [&](auto some) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        const bool in = !decltype(some)::value || s0 + 4 * u < a.kv_split;
        const float w = in ? fast_exp2((ml[u][0] - m) * cmul) : 0.f;
        l = __builtin_fmaf(ml[u][1], w, l);
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = __builtin_fmaf(in ? v[u][e] : 0.f, w, o[e]);
      }
    };
    if (s0 + 4 * (U - 1) < a.kv_split) add(std::false_type{});
    else add(std::true_type{});
  }
  if (wave > 0) {
    float (*slot)[64] = red[wave - 1];
    slot[0][lane] = m;
    slot[1][lane] = l;
#pragma unroll
    for (int e = 0; e < 4; e++) slot[2 + e][lane] = o[e];
  }
  __syncthreads();
  if (wave > 0) return;
  float mm = m;
#pragma unroll
  for (int k = 0; k < 3; k++) mm = fmaxf(mm, red[k][0][lane]);
  const float w0 = fast_exp2((m - mm) * cmul);
  l *= w0;
#pragma unroll
  for (int e = 0; e < 4; e++) o[e] *= w0;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float w = fast_exp2((red[k][0][lane] - mm) * cmul);
    l = __builtin_fmaf(red[k][1][lane], w, l);
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = __builtin_fmaf(red[k][2 + e][lane], w, o[e]);
  }
  if (row >= a.Sq) return;
  const int b = bh / a.N, h = bh % a.N, d = 8 * dr + 4 * g;
  const float inv = l > 0.f ? omul / l : 0.f;
  if (d < a.hd) {
    const typename Elem<T>::V2 t0 = Elem<T>::cvt2(o[0] * inv, o[1] * inv), t1 = Elem<T>::cvt2(o[2] * inv, o[3] * inv);
    const typename Elem<T>::V4 ov = {t0[0], t0[1], t1[0], t1[1]};
    *reinterpret_cast<typename Elem<T>::V4*>((T*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)row * a.o_ss + d) = ov;
  }
  if (dr == 0 && g == 0) a.lse[(int64_t)bh * a.Sq + row] = l > 0.f ? mm * mnat + __logf(l) : -INFINITY;
}

template <typename T, int D, int NW, bool BIAS, bool DROP, int KT, int KG, bool PIPE = false>
static hipError_t launch_fwd_kt(FaArgs a, hipStream_t st) {
  using C = SwzCfg<D>;
  constexpr int QG = 1, RG = NW / KG, BM = 32 * QG * RG;
  a.n_tiles = (a.Sq + BM - 1) / BM;
  if (a.Sk >= 32 * KT && !(tile_offsets_fit(a.k_ss, 32 * KT) && tile_offsets_fit(a.v_ss, 32 * KT))) return hipErrorInvalidPitchValue;
  a.kv_share = split_shares(a.B * a.N, a.Sk, a.hd);
  a.merge_alone = fwd_merge_alone<D, KG>() && a.kv_split <= 1 && (long long)a.n_tiles * a.B * a.N > 256;
  a.first_late = first_tile_late(a.B * a.N, a.n_tiles, visible_row_keys(a.Sq, a.Sk, a.prev_blk, a.next_blk, a.row_prefix), 32 * KT);
  const bool mask_t = BIAS || DROP || a.mask_kind == kMaskDense || a.mask_kind == kMaskTile;
  constexpr size_t biasb = BIAS ? (KT == 4 ? 1024 : QG * 4096) : 0;     // per wave, as in the kernel
  constexpr size_t tiles = 4 * 32 * KT * (size_t)C::PITCH + NW * biasb + (size_t)NW * 2 * DropRowStage<DROP, QG, KT>::BYTES,
                   stage = KG > 1 ? fwd_merge_stats<D, NW, KG>() + (size_t)NW * 512 : (size_t)NW * 32 * (C::DB * 64 + 16);
  static_assert(!fwd_merge_alone<D, KG>() || (size_t)RG * (32 * (C::DB * 64 + 16) + C::DB * 4096 + 512) <= tiles, "the tiles' LDS holds the lone merge");
  constexpr size_t smem = tiles > stage ? tiles : stage;
  static_assert(smem <= 160 * 1024, "the workgroup's LDS must fit the CU's 160 KB");
  auto kern = mask_t ? fa_fwd_kernel<T, D, QG, NW, BIAS, DROP, true, KT, KG, PIPE> : fa_fwd_kernel<T, D, QG, NW, BIAS, DROP, BIAS || DROP, KT, KG, PIPE>;
  hipError_t e = allow_dynamic_lds((const void*)kern, smem);
  if (e != hipSuccess) return e;
  const long long nblk = (long long)a.n_tiles * a.B * a.N;
  hipLaunchKernelGGL(kern, dim3((unsigned)(nblk * (a.kv_split > 1 ? a.kv_split : 1))), dim3(64 * NW), smem, st, a);
  e = hipGetLastError();
  if (e == hipSuccess && a.kv_split > 1) {
    // a full bias is added in natural units, everything else in units of q.k (see the kernel)
    const bool acc_bias = BIAS && KT == 4;
    const bool scaled = BIAS && !acc_bias;
    hipLaunchKernelGGL(fa_fwd_combine_kernel<T>, dim3((unsigned)(nblk * RG * 4 * C::DB)), dim3(256), 0, st, a, RG, (int)C::DB,
                       scaled ? kLog2e : a.scale_log2e, scaled ? 1.0f : a.scale, DROP ? a.inv_keep : 1.0f);
    e = hipGetLastError();
  }
  return e;
}

template <typename T, int D, int NW, int KG, bool BIAS, bool DROP>
static hipError_t launch_fwd_t(const FaArgs& a, hipStream_t st) {
  // K/V stream in tiles of 128 keys where registers and LDS allow (8 waves, D <= 128): twice the
  // matrix work between two barriers, -2 % (causal) to -6 % (full).  A bias tile per wave does not fit beside
  // them; a key-only bias that the DMA can stage is a 256-byte row and does.
  constexpr bool BIG = NW == 8 && D <= 128;
  static_assert(BIG || !BIAS, "the bias variants rest on this choice");
  int seen = visible_row_keys(a.Sq, a.Sk, a.prev_blk, a.next_blk, a.row_prefix);
  if constexpr (KG == 4 && D <= 64) {
    if (a.mask_kind == kMaskCausal && a.Sq < seen) seen = a.Sq;
    if (tile_offsets_fit(a.k_ss, 256) && tile_offsets_fit(a.v_ss, 256) &&
        long_tiles_pay(a.B * a.N, a.Sq, a.Sk, a.hd, seen, a.prev_blk < (a.Sq - 1) / 128))
      return launch_fwd_kt<T, D, NW, BIAS, DROP, 8, KG>(a, st);
  }
  // (with a mask tensor the loop runs where a workgroup sees the causal pattern in it)
  if constexpr (BIG && KG == 1 && D <= 64 && !BIAS && !DROP) {
    if (pipelined_pays(a.Sq, seen, a.mask_kind != kMaskNone || a.next_blk == 0 || a.row_prefix)) return launch_fwd_kt<T, D, NW, false, false, 4, 1, true>(a, st);
  }
  if constexpr (BIG && BIAS) {
    return key_bias_stageable(a) ? launch_fwd_kt<T, D, NW, BIAS, DROP, 4, KG>(a, st) : launch_fwd_kt<T, D, NW, BIAS, DROP, 2, KG>(a, st);
  } else {
    return launch_fwd_kt<T, D, NW, BIAS, DROP, BIG ? 4 : 2, KG>(a, st);
  }
}

// SIDE: 2 = bias and dropout variants, 1 = the dropout variant only (head dims 40, 160, 256)
template <typename T, int D, int NW, int KG, int SIDE>
static hipError_t launch_fwd_q(const FaArgs& a, hipStream_t st) {
  const bool bias = a.alibi != nullptr, drop = a.droprow != nullptr || a.dropcol != nullptr;
#ifndef ACCT_DEV_BUILD
  if constexpr (SIDE == 2) {
    if (bias) return drop ? launch_fwd_t<T, D, NW, KG, true, true>(a, st) : launch_fwd_t<T, D, NW, KG, true, false>(a, st);
  }
  if constexpr (SIDE >= 1) {
    if (drop && !bias) return launch_fwd_t<T, D, NW, KG, false, true>(a, st);
  }
#endif
  if (bias || drop) return hipErrorNotSupported;       // (development build: plain variants only)
  return launch_fwd_t<T, D, NW, KG, false, false>(a, st);
}

// Head dim 256 leaves registers for one wave per SIMD only: 4 waves, no key groups.  Four key groups (64 query rows
// per workgroup) are built without bias and dropout and for 128-key tiles.
template <typename T, int D, int SIDE = 2>
static hipError_t launch_fwd_d(const FaArgs& a, int kg, hipStream_t st) {
  if constexpr (D > 160) {
    return launch_fwd_q<T, D, 4, 1, SIDE>(a, st);
  } else {
    if constexpr (D <= 128) {
      if (kg == 4) return launch_fwd_q<T, D, 8, 4, 0>(a, st);
    }
    return kg == 1 ? launch_fwd_q<T, D, 8, 1, SIDE>(a, st) : launch_fwd_q<T, D, 8, 2, SIDE>(a, st);
  }
}

template <typename T>
hipError_t launch_fwd_elem(const FaArgs& a, int Dr, int kg, hipStream_t st) {
  const int D = head_dim_class(Dr);
  if (D == 128) return launch_fwd_d<T, 128>(a, kg, st);
#ifdef ACCT_DEV_BUILD
  return hipErrorNotSupported;
#else
  if (D == 64) return launch_fwd_d<T, 64>(a, kg, st);
  if (D == 80) return launch_fwd_d<T, 80>(a, kg, st);
  if (D == 40) return launch_fwd_d<T, 40, 1>(a, kg, st);
  if (D == 160) return launch_fwd_d<T, 160, 1>(a, kg, st);
  if (D == 256) return launch_fwd_d<T, 256, 1>(a, kg, st);
  return hipErrorInvalidValue;
#endif
}
template hipError_t launch_fwd_elem<ACCT_ELEM>(const FaArgs& a, int Dr, int kg, hipStream_t st);

}  // namespace acct
