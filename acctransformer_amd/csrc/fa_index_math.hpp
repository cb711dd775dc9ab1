// Integer index arithmetic shared by the gfx950 attention kernels and their launchers: workgroup -> tile
// maps, LDS swizzles, head-dim classes, the query-range split of the dK/dV launch.  No HIP in here: the file
// also compiles with a host compiler, which is how the unit tests reach these functions.
#pragma once
#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define ACCT_HD __host__ __device__ __forceinline__
#else
#define ACCT_HD inline
#endif

namespace acct {

// Workgroup id -> (batch*head, launch rank of the tile; rank 0 is launched first).  Workgroups are
// handed to the 8 XCDs round robin (id % 8), each XCD with its own L2.  With many heads the plain
// "head fastest" order gives every CU of an XCD a different head and nothing is shared; instead the
// heads of an XCD are taken 8 at a time and all tiles of those 8 heads are launched together, so
// that the workgroups streaming the same K/V (or Q/dO) rows run side by side on one L2.
ACCT_HD void wg_map(int id, int BH, int n_tiles, int& bh, int& rank) {
  if (BH > 64 && (BH & 63) == 0) {
    const int xcd = id & 7, slot = id >> 3;
    const int per_group = 8 * n_tiles;
    const int grp = slot / per_group, r = slot - grp * per_group;
    rank = r >> 3;
    bh = xcd + 8 * (grp * 8 + (r & 7));
  } else {
    bh = id % BH;
    rank = id / BH;
  }
}

// Position of workgroup `id` of `n` in an order in which each XCD has one contiguous eighth (of those it is handed, id % 8).
ACCT_HD int xcd_span(int id, int n) {
  const int per = n / 8, rem = n % 8, xcd = id & 7;
  return xcd * per + (xcd < rem ? xcd : rem) + (id >> 3);
}

// Workgroup id of a forward launch over `split` key slices -> slice and the id that wg_map takes.  The row tiles of one head
// and slice read the same keys.  `share`: they follow each other on one XCD, whose L2 then fetches them once; in the plain order,
// slice by slice, they sit on different XCDs.  (Above 64 heads in wg_map's other order a split launch has one row tile per head.)
//
// In the plain order a head's tiles sit on one XCD anyway where the heads are a multiple of 8: nothing to gain there (1.00 to
// 1.04 of the plain time).  Otherwise sharing pays once K and V no longer fit the eight L2s (32 MB, less what else passes
// through).  Time shared / plain, 1 to 7 heads (4 heads, whose tiles sit on two XCDs, gain half), 256 / 512 / 1024 queries; a
// pass that finds K and V in the caches: 5 million elements of K D64 1.09 / 1.04 / 0.98, D128 1.06 / 1.01 / 0.96; 6: 1.06 / 1.01 / 0.99,
// 1.03 / 0.95 / 0.95; 7: 1.00 / 0.97 / 0.97, 0.97 / 0.95 / 0.95; 9: 0.98 / 0.97 / 0.96, 0.96 / 0.95 / 0.94; 16: 0.97 / 0.94 / 0.93, 0.95 /
// 0.92 / 0.92; 32: 0.96 / 0.93 / 0.93, 0.94 / 0.91 / 0.92; from memory 0.91 to 1.04, 0.97 on average.  1 head, 256 x 131072, D128 34.5 / 32.9 us;
// 2, 500 x 100000, D64 45.9 / 43.2; 5, 400 x 30000, D128 55.8 / 49.3.
ACCT_HD bool split_shares(int BH, int Sk, int D) { return BH % 8 != 0 && (long long)BH * Sk * D >= 7000000; }
ACCT_HD void split_map(int id, int BH, int n_tiles, int split, bool share, int& slice, int& wg) {
  const int n_wg = BH * n_tiles;
  if (!share || n_tiles == 1 || (BH > 64 && (BH & 63) == 0)) {
    slice = id / n_wg;
    wg = id - slice * n_wg;
    return;
  }
  const int at = xcd_span(id, n_wg * split), pair = at / n_tiles, rank = at - pair * n_tiles;
  slice = pair / BH;
  wg = rank * BH + (pair - slice * BH);
}

// A tile of `rows` rows of 2-byte elements is addressed by a base and 32-bit byte offsets: whether the last row's fit (a row
// has up to 256 elements).  Launchers refuse what does not: a test in the kernels cost the triangle layer's forward 0.6 %.
ACCT_HD bool tile_offsets_fit(int64_t row_stride, int rows) { return row_stride * (rows - 1) <= 0x7fffffffll - 256; }
// Row strides of a backward end here (its tiles have 64 rows; in whole chunks of 8 elements).
constexpr int64_t kBwdRowStrideEnd = 34087040;

// ---- swizzle of the LDS tiles that the direct-to-LDS loads fill ----
// Row pitch is a power of two (no padding, as the DMA writes 64 consecutive 16-byte
// slots per wave instruction); the 16-byte chunk c of row r lives in slot c ^ swz(r).
// The LDS serves a 16-byte read in groups of 16 lanes over 64 four-byte banks, so the
// fragment reads (lane = row) need the 16 rows of a group in 16 different slots of the
// 256 bytes the banks span: measured 4.3 clocks per wave instruction against 8.2 when
// only eight rows differ.  For 256-byte rows that is a four-bit swizzle,
// swz(r) = ((r & 3) << 1) | ((r >> 2) & 1) | (r & 8); its low three bits also put one
// 32-byte chunk PAIR of four consecutive rows into four different pairs of slots, which
// is what the transposed 8-byte reads (4 rows x 32 bytes per 16 lanes) need.  For
// 128-byte rows two consecutive rows span the banks and swz(r) = (r >> 1) & 7.
ACCT_HD int swz3(int row) { return ((row & 3) << 1) | ((row >> 2) & 1); }

template <int D> struct SwzCfg {
  static constexpr int KS = (D + 15) / 16;      // 16-wide k-steps across the head dim (the last one half empty when D % 16 == 8)
  static constexpr int DB = (D + 31) / 32;      // 32-wide blocks across the head dim
  static constexpr int CPR = D / 8;             // valid 16-byte chunks per row
  static constexpr int CH = D <= 64 ? 8 : (D <= 128 ? 16 : 32);   // chunk slots per LDS row
  static constexpr int PITCH = CH * 16;
  static constexpr int RPI = 64 / CH;           // rows covered by one wave-wide DMA instruction
  // (rows of 512 bytes wrap around the banks twice: the four-bit swizzle of the 256-byte rows serves them too)
  static ACCT_HD int swz(int row) { return CH >= 16 ? (swz3(row) | (row & 8)) : ((row >> 1) & 7); }
  // Transposed reads come in pairs, rows r..r+3 and r+8..r+11 with r % 16 < 8: the second row group has
  // the top swizzle bit set, so its slot differs in that bit.  Which way depends only on the 32-column
  // block db the read belongs to (chunk 4 db + 0..3), i.e. the distance is a compile-time constant.
  static constexpr int tr_hi(int db) {
    return 8 * PITCH + (CH >= 16 ? (((db >> 1) & 1) ? -128 : 128) : ((db & 1) ? -64 : 64));
  }
};

// idx / n for idx < 1024 and n <= 32 (the epilogues' chunk index -> row): exact with a 16-bit reciprocal
ACCT_HD int div_small(int idx, uint32_t inv16) { return (int)(((uint32_t)idx * inv16) >> 16); }
ACCT_HD uint32_t recip16(int n) { return (65536u + (uint32_t)n - 1u) / (uint32_t)n; }

// byte offset of logical chunk `lc` in a row whose swz3(row) is `swz`
ACCT_HD int swz_off(int lc, int swz) { return (lc ^ swz) << 4; }

// The keep bits by key column (FaArgs::dropcol), [B*N, Tr, Sk] entries of four 32-bit words: index of the first word of an
// entry, and the byte offset of word `w` of the entry `dk` keys after it.  A workgroup addresses the entries of its keys
// as a 64-bit base for its first one and such an offset per lane, which stays below 4 KB whatever Sk is.
ACCT_HD int64_t keep_col_entry(int64_t bh, int Tr, int qb, int Sk, int key) { return ((bh * Tr + qb) * Sk + key) * 4; }
ACCT_HD uint32_t keep_col_offset(int dk, int w) { return (uint32_t)dk * 16u + (uint32_t)w * 4u; }

// The kernels are built for the head dims 40, 64, 80, 128, 160 and 256.  Any other multiple of 8 runs on the next
// built size of its row layout (128-, 256- or 512-byte LDS rows): the columns past the head dim are never loaded
// as operands (zero fragments) and never stored.
ACCT_HD int head_dim_class(int D) {
  if (D == 40 || D == 80 || D == 160) return D;
  return D <= 64 ? 64 : (D <= 128 ? 128 : 256);
}

// With few heads and a short key sequence (cross attention on 77 keys) the dK/dV kernel's key tiles are a handful of
// workgroups for 256 CUs: the query range is then cut into q_split slices that run side by side, and a second kernel
// adds their sums.  The split of a launch whose waves own two key groups (256 keys per workgroup, 128 above head dim
// 128): as many slices as fill the CUs, at least 512 query rows each.
// Returns q_split (1 = no split) and the bytes of workspace the slices' sums take.
// `n_cu`: compute units of the device that runs the launch; the workspace-size query passes the 256 of a whole
// MI355X, which is also the upper bound of what a partition of it asks for.
struct DkdvSplit { int q_split; size_t part_bytes; };
ACCT_HD size_t dkdv_part_bytes(int B, int N, int Sk, int D, int ngk, int split) {
  const int db = (head_dim_class(D) + 31) / 32;
  const long long n_wg = (long long)B * N * ((Sk + 128 * ngk - 1) / (128 * ngk));
  return split > 1 ? (size_t)split * (size_t)n_wg * 8 * ngk * db * 1024 * sizeof(float) : 0;
}
ACCT_HD DkdvSplit dkdv_split(int B, int N, int Sq, int Sk, int D, int n_cu = 256) {
  const int ngk = head_dim_class(D) > 128 ? 1 : 2;
  const long long n_wg = (long long)B * N * ((Sk + 128 * ngk - 1) / (128 * ngk));
  const long long tiles64 = (Sq + 63) / 64;
  long long s = (n_cu > 256 ? 256 : n_cu) / n_wg;
  if (tiles64 / 8 < s) s = tiles64 / 8;              // a slice keeps at least 512 query rows
  if (s > 16) s = 16;
  if (s < 2) return {1, 0};
  return {(int)s, dkdv_part_bytes(B, N, Sk, D, ngk, (int)s)};
}

// How the dK/dV kernel cuts its work: ngk 32-key groups per wave (4 * 32 * ngk keys per workgroup) and q_split slices
// of the query range.  One key group per wave does half the work of two in 0.65 of the time (every Q / dO fragment
// read from LDS feeds one MFMA instead of two), or in 0.53 where the head dim lets several workgroups share a CU, so
// it pays where its finer units fill the last round better.  The estimate below prices the candidates in microseconds:
// steps of 32 query rows, rounds of workgroups, and for slices the second launch and the sums written and read.
// Measured, two groups / one group (us): 96 heads, 1000 x 1000, D64 93.6 / 74.4; 24, 3000 x 3000, D64 250 / 196;
// 16, 4096 x 4096, D64 (256 and 512 workgroups: no round to save) 158 / 173; 144, 285 x 285, D128 47.5 / 33.8;
// 80, 2000 x 2000, D128 378 / 394; causal: 64, 2048 x 2048, D128 154 / 177; 24, 2424 x 2424, D128 165 / 120.
// With slices, before / now: 32 heads, 1024 x 77, D80 44.2 (two groups, 2 slices) / 26.1 (one group, 4); 40, 1611 x 77,
// D160 43.7 (6) / 39.4 (4).
//
// A band lets 128 keys see only `blocks` of the 128-row blocks (`share` of that on average; all of them in the
// `whole` part of the sequence, less at its ends), so 128 * ngk keys are walked by blocks + ngk - 1 of them and finer units
// pass fewer rows that their keys do not see.  Backward of a launch with two groups / one group: 64 heads, S4096, D64, one
// block back 144.5 / 117.8 us; 32, S2048, D128, eight back 128.6 / 143.6; 48, S1500, D80 (288 and 576 workgroups, of which
// 168 and 336 are whole), five back 78.9 / 86.4; 24, S2048, D128 (192 and 384), four back 81.6 / 89.1.
struct RowBand { bool on; int blocks; double share, whole; };
ACCT_HD RowBand row_band(int Sq, int prev_blk, int next_blk) {
  const int T = (Sq + 127) / 128, p = prev_blk < T ? prev_blk : T - 1, q = next_blk < T ? next_blk : T - 1;
  const double all = (double)T * (1 + p + q);
  return {p + q + 1 < T, 1 + p + q, (all - 0.5 * p * (p + 1.0) - 0.5 * q * (q + 1.0)) / all, (double)(T - p - q) / T};
}
struct DkdvPlan { int ngk, q_split; size_t part_bytes; };
ACCT_HD double dkdv_estimate(int B, int N, int Sq, int Sk, int D, bool tri, int ngk, int split, int n_cu, int prev_blk, int next_blk) {
  const int dc = head_dim_class(D);
  const double n = (double)B * N * ((Sk + 128 * ngk - 1) / (128 * ngk)) * split;
  const RowBand band = row_band(Sq, prev_blk, next_blk);
  int steps = 2 * (((Sq + 63) / 64 + split - 1) / split);
  if (band.on && band.blocks + ngk - 1 < steps / 4) steps = 4 * (band.blocks + ngk - 1);
  double walk = steps * (0.62 + 0.0037 * dc) * (ngk == 2 ? 1 / 0.65 : 1.0);
  if (ngk == 1 && dc <= 64 && n > n_cu) walk *= 0.53 / 0.65;
  double rounds = (double)(((long long)n + n_cu - 1) / n_cu);
  if (tri) {   // below the causal diagonal half of the workgroups' steps are absent, the heaviest start first
    // (on long walks up to twice as many workgroups as CUs end together, the light ones beside the heaviest; shorter ones do
    // not.  D64, two groups / one group: 32 heads, S4096 (512 and 1024 workgroups) backward 287 / 302 us, S3500 (448 and 896)
    // 223 / 232, 40 heads, S3000 (480 and 960) 215 / 219; but 80 heads, S1500 (480 and 960) 133 / 128)
    rounds = 0.5 * n / n_cu + 0.3;
    if (steps > 80 && split == 1 && n <= 2 * n_cu && rounds > 1.06) rounds = 1.06;
    if (rounds < 1.0) rounds = 1.0;
  } else if (band.on) {   // the workgroups at the ends of the band are shorter than the rest
    const double whole = (double)(((long long)(band.whole * n) + n_cu - 1) / n_cu), r = band.share * n / n_cu + 0.3;
    rounds = r < whole ? whole : r < rounds ? r : rounds;
  }
  return 8.0 + walk * rounds + (split > 1 ? 6.5 + 2e6 / 6e12 * (double)dkdv_part_bytes(B, N, Sk, D, ngk, split) : 0.0);
}
// `room`: bytes of workspace there are for the slices' sums; `tri`: key blocks after the query's block are left out;
// `prev_blk`, `next_blk`: the band
ACCT_HD DkdvPlan dkdv_plan(int B, int N, int Sq, int Sk, int D, bool tri, size_t room, int n_cu = 256, int prev_blk = 65536, int next_blk = 65536) {
  const bool wide = head_dim_class(D) > 128;           // (one key group per wave is all the registers hold)
  DkdvPlan best = {wide ? 1 : 2, 1, 0};
  double t_best = dkdv_estimate(B, N, Sq, Sk, D, tri, best.ngk, 1, n_cu, prev_blk, next_blk);
  const DkdvSplit two = dkdv_split(B, N, Sq, Sk, D, n_cu);
  if (!wide && two.q_split > 1 && two.part_bytes <= room) {
    const double t = dkdv_estimate(B, N, Sq, Sk, D, tri, 2, two.q_split, n_cu, prev_blk, next_blk);
    if (t < t_best) { t_best = t; best = {2, two.q_split, two.part_bytes}; }
  }
  const double n1 = (double)B * N * ((Sk + 127) / 128);
  const bool banded = row_band(Sq, prev_blk, next_blk).on;
  for (int s = 1; s <= 16 && s <= (Sq + 63) / 64 && (s == 1 || n1 * s <= (tri ? 2.0 : 1.0) * n_cu); s *= 2) {
    const size_t bytes = dkdv_part_bytes(B, N, Sk, D, 1, s);
    const double t = dkdv_estimate(B, N, Sq, Sk, D, tri, 1, s, n_cu, prev_blk, next_blk);
    if (bytes <= room && t < (banded ? 0.9 : s > 1 ? 0.95 : 1.0) * t_best) { t_best = t; best = {1, s, bytes}; }
  }
  return best;
}

// Keys that the 128-row block with the longest walk sees: the band (blocks qb - prev_blk .. qb + next_blk) and the row
// prefix, whose last group sees the most, bound it; the caller's Sk bounds it as well.
ACCT_HD int visible_row_keys(int Sq, int Sk, int prev_blk, int next_blk, int row_prefix) {
  const long long qb_last = (Sq - 1) / 128, kb_last = (Sk - 1) / 128;
  const long long before = prev_blk < qb_last ? prev_blk : qb_last, after = next_blk < kb_last ? next_blk : kb_last;
  long long keys = (before + 1 + after) * 128;
  if (row_prefix > 0 && ((long long)(Sq - 1) / row_prefix + 1) * row_prefix < keys) keys = ((long long)(Sq - 1) / row_prefix + 1) * row_prefix;
  return keys < Sk ? (int)keys : Sk;
}

// Keys that a row sees on average.  `one_sided`: what it sees ends with the row (causal, a band that ends at the query's block,
// a row prefix).
ACCT_HD long long mean_row_keys(int Sq, int row_keys, bool one_sided) {
  if (!one_sided) return row_keys;
  return row_keys >= Sq ? ((long long)Sq + 1) / 2 : row_keys - (long long)row_keys * row_keys / (2ll * Sq);
}
// The forward's pipelined tile loop (fa_fwd.hip, head dims up to 64) takes 3 to 6 % off a tile's step, but the first scores and the
// last product have nothing beside them: about one step, with its wait and barrier, more per workgroup.  Forward, us, plain /
// pipelined: 256 heads, 2048 x 128 keys, D64 48 / 56; x 512 102 / 109; x 768 141 / 144; x 1024 178 / 179; x 1536 258 / 255; x 3000
// 506 / 478; x 8192 1295 / 1243; D40 39 / 46; 92 / 93; 125 / 128; 160 / 162; 235 / 226; 460 / 427; 1172 / 1127.  16 heads, 4096 rows are alike.
// Causal: 256 heads, S1024, D40 52.9 / 54.7; S1536 108 / 109; S2048 176 / 173; S4096 640 / 623; 32 heads, S2048 35.6 / 33.5.
ACCT_HD bool pipelined_pays(int Sq, int row_keys, bool one_sided) { return mean_row_keys(Sq, row_keys, one_sided) >= 1024; }

// Four key groups leave a wave 32 keys of a 128-key tile: a step of latencies.  At head dims up to 64 LDS has room for 256-key
// tiles, one workgroup to a CU, and a step of those takes 1.65 times as long.  They pay where the longest walk has that much fewer
// of them: forward, 128 / 256 keys, us, D64, 4 heads, 512 queries x 129 keys 5.9 / 5.6; 257 (3 and 2 tiles) 6.7 / 7.0; 384 6.5 / 6.9; 512
// 7.3 / 6.7; 600 (5 and 3) 8.5 / 8.4; 768 9.0 / 8.1; 1000 11.0 / 10.0; 64 x 512 causal (1 and 1) 4.7 / 5.2; a band of two blocks (2 and 2,
// where it starts within a tile) 5.7 / 6.2.  Not where every workgroup has keys of its own from memory: 250 heads, 64 x 500 (32 MB
// of K and V, what the eight L2s hold) 8.5 / 8.2; x 600 10.3 / 11.1; x 1024 13.7 / 14.3 (D40, 41 MB: 11.0 / 10.3).  Nor in more than one
// round: 20 heads, 1024 x 1024 causal, 320 workgroups 12.2 / 12.7.
// `seen`: keys of the longest walk; `moving`: walks that start at any block.
ACCT_HD bool long_tiles_pay(int BH, int Sq, int Sk, int D, int seen, bool moving) {
  const int n128 = (seen + 127) / 128, n256 = moving ? n128 / 2 + 1 : (n128 + 1) / 2;
  const bool own_keys = Sq <= 64 && D > 40 && (long long)BH * Sk * D > (8 << 20);
  return (long long)BH * ((Sq + 63) / 64) <= 256 && !own_keys && 20 * n128 > 33 * n256;
}

// Whether the forward requests its first tile behind the Q fragments and not ahead of them: launches of more than one round
// whose workgroups walk a single tile and have a head's rows to themselves (nothing is left to do meanwhile, and Q waits behind
// K and V).  Forward, us, ahead / behind, 1024 heads: 77 x 77, D128 31.5 / 29.1; 128 x 128 39.5 / 37.2; 256 x 128 48.7 / 47.2; with
// dropout 53.4 / 49.4; D80 128 x 128 26.5 / 25.3; D64 18.0 / 16.8, dropout 26.2 / 23.8.  Where the row tiles of a head share its
// keys it is the other way round: 1024 x 77, D128 174 / 188; D80 124 / 134.  (Head dims 40, 160 and 256: level or 1 to 3 % slower.)
// `seen`: keys that a workgroup's rows see.
ACCT_HD bool first_tile_late(int BH, int n_tiles, int seen, int tile_keys) { return n_tiles == 1 && BH > 256 && seen <= tile_keys; }

// How the forward kernel cuts its work.  kg: key groups of the workgroup (fa_fwd.hip; 256 / kg query rows per
// workgroup).  kv_split: slices of the key range on workgroups of their own, which a second kernel adds up (1: none).
//
// A workgroup of kg = 4 steps through its key tiles 2.2 times as fast as one of kg = 1 (1.22 against 2.68 us per 128
// keys at head dim 128, each alone on its CU) but does a quarter of the work, so kg > 1 pays only where its larger
// number of workgroups still runs in one round: B1 N16 S1024 D64 (64 / 128 / 256 workgroups) 20.2 / 14.5 / 11.7 us
// for kg 1 / 2 / 4, N20 (80 / 160 / 320) 20.3 / 14.8 / 16.6, N40 (160 / 320 / 640) 20.9 / 21.8 / 24.3.  Below the
// causal diagonal (`tri`) half of the workgroups are light and one and a quarter (kg 4) or, over long rows, two
// (kg 2) times the CUs still pay: N24 S2048 D128 (192 / 384 / 768) 50.1 / 36.3 / 51.0, but N96 S512 18.3 / 20.0 / 28.3.
//
// The slices cost a second launch and the slices' sums written and read (about 6.5 us, and 3 TB/s); they are
// taken where the estimate below says that the shorter walk saves more: 1 head, 256 queries x 131072 keys
// 1253 -> 37 us; 8 heads, 512 x 8192 80 -> 33; not for 4 heads, 2048 x 2048 causal (24.8 against 28.9).
// Their number is a power of two or as many as the CUs hold, whichever walks least; powers of two alone leave up to
// half of the CUs idle.  With / without the latter: 3 heads, 300 x 60000, D128 (28 / 16 slices) 54.2 / 75.0 us; 5 heads,
// 400 x 60000, D64 (12 / 8) 67.6 / 88.1; 40 heads, 1 x 8000, D64 (6 / 4) 24.1 / 29.7; 7 heads, 500 x 20000 (9 / 8) 57.8 / 58.2.
struct FwdPlan { int kg, kv_split; size_t part_bytes; };
ACCT_HD size_t fwd_part_bytes(int B, int N, int Sq, int D, int kg, int split) {
  const int dc = head_dim_class(D), rows = dc > 160 ? 128 : 256 / kg;
  const long long groups = (long long)B * N * ((Sq + rows - 1) / rows) * (rows / 32);     // of 32 query rows
  return split > 1 ? (size_t)split * (size_t)groups * ((dc + 31) / 32 * 1024 + 64) * sizeof(float) : 0;
}
// A launch that fills the chip more than once still ends in a round that may be nearly empty.  Workgroups of half the
// rows take `half` of the time of a whole one; true when their rounds add up to less.  Forward, kg 1 / 2 (us): 96 heads,
// 1000 x 1000, D64 (384 / 768 workgroups) 42.5 / 37.0; 24, 3000 x 3000, D64 (288 / 576) 109.5 / 86.6; 144, 285 x 285, D128
// (288 / 432) 25.3 / 22.6; but 96, 1000 x 1000, D128 (2 and 3 rounds of 0.7) 64.5 / 67.9; 16, 4096 x 4096, D64 (256 / 512) 80 / 84.
ACCT_HD bool half_workgroups_pay(long long n1, long long n2, int n_cu, double half) {
  return (double)((n2 + n_cu - 1) / n_cu) * half < 0.97 * (double)((n1 + n_cu - 1) / n_cu);
}
// `side`: a bias or dropout (not built for kg = 4); `tri`: key blocks after the query's block are left out;
// `can_split`: there is room for the slices' sums; `row_keys`: keys that the widest row block sees (visible_row_keys) --
// what the slices are cut from; `one_sided`: a band that ends at the query's block, where the workgroups at one end are
// short and whole rounds do not count (48 heads, S1500, D64, five blocks back 19.6 us for kg 1, 22.6 for kg 2)
ACCT_HD FwdPlan fwd_plan(int B, int N, int Sq, int Sk, int D, bool side, bool tri, bool can_split, int n_cu = 256, int row_keys = 0x7fffffff,
                         bool one_sided = false) {
  const int dc = head_dim_class(D);
  const long long bh = (long long)B * N, n1 = bh * ((Sq + 255) / 256), n2 = bh * ((Sq + 127) / 128), n4 = bh * ((Sq + 63) / 64);
  int kg = 1;
  if (dc <= 128 && !side && n4 <= (tri ? n_cu + n_cu / 4 : n_cu)) kg = 4;
  else if (dc <= 160 && (n2 <= n_cu || (tri && n1 < n_cu && Sk >= 1024))) kg = 2;
  else if (dc <= 128 && !tri && !one_sided && half_workgroups_pay(n1, n2, n_cu, dc <= 64 ? 0.55 : 0.7)) kg = 2;
  // slices: microseconds of a workgroup's walk against those of a slice's, plus the second launch and the traffic
  const int kg_s = dc > 160 ? 1 : 2;
  const long long n_s = kg_s == 2 ? n2 : bh * ((Sq + 127) / 128);
  int seen = tri && Sq < Sk ? Sq : Sk;
  if (row_keys < seen) seen = row_keys;
  const int tiles = (seen + 127) / 128;
  const double per_tile = 0.5 + 0.72 / 128 * dc;                       // kg = 4; 1.3 and 2.2 times that for kg = 2 and 1
  double best = per_tile * (kg == 4 ? 1.0 : kg == 2 ? 1.3 : 2.2) * tiles;
  int split = 1;
  const long long fit = n_cu / n_s < 256 ? n_cu / n_s : 256;
  const int most = fit < tiles ? (int)fit : tiles;
  for (int i = 2; can_split && most >= 2; i *= 2) {                    // 2, 4, 8 ... and as many as there are CUs for
    const int cut = i < most ? i : most, walk = (tiles + cut - 1) / cut, s = (tiles + walk - 1) / walk;
    const double t = per_tile * (kg_s == 2 ? 1.3 : 2.2) * walk + 6.5 + 2e6 / 3e12 * (double)fwd_part_bytes(B, N, Sq, D, kg_s, s);
    if (t < best) { best = t; split = s; }
    if (i >= most) break;
  }
  if (split > 1) kg = kg_s;
  return {kg, split, fwd_part_bytes(B, N, Sq, D, kg, split)};
}

// The forward with one query row per head (fa_fwd_row.hip): parts of the key range per head, each a workgroup of its own,
// which a second kernel adds up (1: none).  A workgroup alone takes 1.1 us per batch of 64 KB of K and V, a little more the more
// others there are, those that share a CU 1.8; all of them together 1 us per 6.6 MB; 95 of them start per us; the second kernel
// takes 3.4 us and more.
// One part / the parts taken (us; bf16): 8 heads, 512 keys, D128 7.3 / 7.3 (4 parts 7.9); 8, 8192, D128 75 / 13.7 (16); 64, 2048,
// D64 13.7 / 12.1 (2); 96, 8192, D128 88 / 65 (2); 256, 8192, D128 157 / 157 (2 parts 160); 512, 128, D64 6.8 / 6.8 (2 13.4).
struct RowPlan { int parts; size_t part_bytes; };
ACCT_HD int row_batch(int D) { return D <= 64 ? 256 : D <= 128 ? 128 : 64; }             // keys
ACCT_HD size_t row_part_bytes(int B, int N, int D, int parts) {
  return parts > 1 ? (size_t)parts * (size_t)B * N * (D + 2) * sizeof(float) : 0;
}
ACCT_HD RowPlan row_plan(int B, int N, int keys, int D, bool can_split) {
  const double heads = (double)B * N, stream = heads * keys * D * 4 / 6.6e6;
  const int batches = (keys + row_batch(D) - 1) / row_batch(D);
  int best = 1;
  double t_best = 0;
  for (int parts = 1; parts <= 256 && parts <= batches && (parts == 1 || can_split); parts *= 2) {
    const double n = heads * parts, walk = (double)((batches + parts - 1) / parts);
    double t = walk * (1.12 + 0.002 * (n < 256 ? n : 256));
    if (n > 256) t = walk * 1.82 * (double)(((long long)n + 255) / 256);                 // several workgroups share some CUs
    if (stream > t) t = stream;
    if (n / 95 > t) t = n / 95;
    if (parts > 1) t += 3.4 + 0.02 * parts;
    if (parts == 1 || t < t_best) { t_best = t; best = parts; }
  }
  return {best, row_part_bytes(B, N, D, best)};
}

// Key groups of the dQ kernel (fa_bwd.hip): 2 where 256-row workgroups would leave CUs idle.  A workgroup of half the
// rows takes 0.6 to 0.75 of the time, so it pays in one round only: 8 heads, S3728, D128 causal 175 -> 112 us; 16 heads,
// 1024 x 1024, D128 with dropout 47.9 -> 33.4; 24 heads, S2424, D128 causal 116 -> 90; but 80 heads, 2000 x 2000 272 / 277
// and 16 heads, 4096 x 4096, D64 107 / 124.
ACCT_HD int dq_key_groups(int B, int N, int Sq, int Sk, int D, bool tri, int n_cu = 256) {
  const int dc = head_dim_class(D);
  if (dc > 128) return 1;
  const long long bh = (long long)B * N, n1 = bh * ((Sq + 255) / 256), n2 = bh * ((Sq + 127) / 128);
  return n2 <= n_cu || (tri && n1 < n_cu && Sk >= 1024) ? 2 : 1;
}

}  // namespace acct
