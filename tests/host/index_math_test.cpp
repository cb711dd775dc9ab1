// Host-compiled unit tests of the integer index arithmetic the gfx950 kernels rest on
// (acctransformer_amd/csrc/fa_index_math.hpp).  Built and run by tests/test_index_math.py with g++;
// prints one line per failed check and exits with the number of failures.
// Test tier modelled on the reference's helper-level unit tests
// (tests/train/flash_attention/ut/test_split_core_strategy.py, test_tensor_transformat.py).
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <set>
#include <vector>

#include "../../acctransformer_amd/csrc/fa_index_math.hpp"

using namespace acct;

static int failures = 0;
#define CHECK(cond, ...)                                   \
  do {                                                     \
    if (!(cond)) {                                         \
      if (failures < 20) { printf("FAIL %s:%d: ", __FILE__, __LINE__); printf(__VA_ARGS__); printf("\n"); } \
      failures++;                                          \
    }                                                      \
  } while (0)

// every (batch*head, tile rank) pair is produced by exactly one workgroup id, whichever branch of the map runs
static void test_wg_map() {
  const int tiles[] = {1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64};
  std::vector<char> seen;
  for (int BH = 1; BH <= 512; BH++)
    for (int nt : tiles) {
      seen.assign((size_t)BH * nt, 0);
      bool ok = true;
      for (int id = 0; id < BH * nt && ok; id++) {
        int bh = -1, rank = -1;
        wg_map(id, BH, nt, bh, rank);
        ok = bh >= 0 && bh < BH && rank >= 0 && rank < nt && !seen[(size_t)bh * nt + rank];
        if (ok) seen[(size_t)bh * nt + rank] = 1;
      }
      CHECK(ok, "wg_map is not a bijection for BH=%d n_tiles=%d", BH, nt);
    }
  // the grouped branch: the workgroups of one head all carry the same id % 8 (one XCD, one L2), ranks ascend with the id
  for (int BH : {128, 256, 512}) {
    const int nt = 16;
    std::vector<int> xcd(BH, -1), last_rank(BH, -1);
    for (int id = 0; id < BH * nt; id++) {
      int bh, rank;
      wg_map(id, BH, nt, bh, rank);
      CHECK(xcd[bh] < 0 || xcd[bh] == (id & 7), "head %d of BH=%d is spread over XCDs", bh, BH);
      xcd[bh] = id & 7;
      CHECK(rank > last_rank[bh], "ranks of head %d do not ascend with the workgroup id", bh);
      last_rank[bh] = rank;
    }
  }
  // the plain branch: head index fastest
  {
    int bh, rank;
    wg_map(64 * 3 + 5, 64, 8, bh, rank);
    CHECK(bh == 5 && rank == 3, "plain branch: got bh=%d rank=%d", bh, rank);
  }
}

// A 16-byte fragment read is served 16 lanes at a time; the 16 rows of such a group must land in 16 different
// 16-byte slots of the 256 bytes the banks span, for every logical chunk.
template <int D> static void test_swizzle_rows() {
  using C = SwzCfg<D>;
  for (int r0 = 0; r0 < 64; r0 += 16)
    for (int c = 0; c < C::CH; c++) {
      std::set<int> slots;
      for (int r = r0; r < r0 + 16; r++) {
        const int addr = r * C::PITCH + ((c ^ C::swz(r)) << 4);
        CHECK(((c ^ C::swz(r)) >= 0) && ((c ^ C::swz(r)) < C::CH), "D=%d: chunk %d of row %d leaves the row", D, c, r);
        slots.insert((addr % 256) / 16);
      }
      CHECK(slots.size() == 16, "D=%d rows %d..%d chunk %d: %zu distinct bank slots", D, r0, r0 + 15, c, slots.size());
    }
  // the swizzle is a permutation of a row's chunks and repeats every 16 rows
  for (int r = 0; r < 64; r++) {
    std::set<int> s;
    for (int c = 0; c < C::CH; c++) s.insert(c ^ C::swz(r));
    CHECK((int)s.size() == C::CH, "D=%d row %d: the swizzle is not a permutation", D, r);
    CHECK(C::swz(r) == C::swz(r + 16), "D=%d: the swizzle does not repeat after 16 rows at row %d", D, r);
  }
}

// Transposed reads: the lanes of a wave address rows trow = 4 g + (lane % 16) / 4 (g = lane / 32) of an 8-row group,
// chunk 4 db + tchunk; the partner read of rows + 8 must sit exactly tr_hi(db) bytes further, for every lane and db.
template <int D> static void test_tr_hi() {
  using C = SwzCfg<D>;
  for (int lane = 0; lane < 64; lane++) {
    const int g = lane >> 5;
    const int trow = 4 * g + ((lane & 15) >> 2);
    const int tchunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    for (int db = 0; db < C::DB; db++)
      for (int grp = 0; grp < 64; grp += 16) {
        const int lo = (grp + trow) * C::PITCH + swz_off(4 * db + tchunk, C::swz(grp + trow));
        const int hi = (grp + trow + 8) * C::PITCH + swz_off(4 * db + tchunk, C::swz(grp + trow + 8));
        CHECK(hi - lo == C::tr_hi(db), "D=%d lane %d db %d: rows +8 sit %d bytes away, tr_hi says %d", D, lane, db, hi - lo, C::tr_hi(db));
      }
  }
  // the four rows x two 16-byte chunks that a 16-lane group of a transposed read touches fall into 8 different slots
  // (256- and 512-byte rows; with 128-byte rows two consecutive rows share a swizzle value and the eight pieces
  // fall into 4 slots, a two-way conflict that the head dims up to 64 live with)
  for (int db = 0; db < C::DB; db++)
    for (int half = 0; half < 2; half++)
      for (int g = 0; g < 2; g++) {
        std::set<int> slots;
        for (int i = 0; i < 16; i++) {
          const int lane = 32 * g + 16 * half + i;
          const int trow = 4 * g + ((lane & 15) >> 2), tchunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
          const int addr = trow * C::PITCH + swz_off(4 * db + tchunk, C::swz(trow));
          slots.insert((addr % 256) / 16);
        }
        const size_t want = C::CH >= 16 ? 8 : 4;
        CHECK(slots.size() == want, "D=%d db %d: a transposed 16-lane group touches %zu slots, expected %zu", D, db, slots.size(), want);
      }
}

static void test_head_dim_class() {
  const int built[] = {40, 64, 80, 128, 160, 256};
  for (int D = 8; D <= 256; D += 8) {
    const int c = head_dim_class(D);
    bool is_built = false;
    for (int b : built) is_built |= b == c;
    CHECK(is_built && c >= D, "head dim %d runs on %d", D, c);
    // same LDS row layout: 128-, 256- or 512-byte rows
    auto layout = [](int d) { return d <= 64 ? 0 : (d <= 128 ? 1 : 2); };
    CHECK(layout(c) == layout(D), "head dim %d (layout %d) runs on %d (layout %d)", D, layout(D), c, layout(c));
    for (int b : built) CHECK(!(b >= D && b < c && layout(b) == layout(D) && (b == D)), "head dim %d skips its own built size", D);
  }
  CHECK(head_dim_class(40) == 40 && head_dim_class(48) == 64 && head_dim_class(72) == 128 && head_dim_class(136) == 256, "class table");
}

static void test_dkdv_split() {
  for (int B : {1, 2, 4, 16})
    for (int N : {1, 4, 16, 32})
      for (int Sq : {64, 511, 512, 1024, 4096, 131072})
        for (int Sk : {1, 77, 128, 256, 257, 2048})
          for (int D : {40, 64, 128, 160, 256})
            for (int n_cu : {32, 64, 256, 304}) {
              const DkdvSplit sp = dkdv_split(B, N, Sq, Sk, D, n_cu), full = dkdv_split(B, N, Sq, Sk, D);
              const int ngk = head_dim_class(D) > 128 ? 1 : 2, db = (head_dim_class(D) + 31) / 32;
              const long long n_wg = (long long)B * N * ((Sk + 128 * ngk - 1) / (128 * ngk));
              CHECK(sp.q_split >= 1 && sp.q_split <= 16, "q_split %d out of range", sp.q_split);
              CHECK(sp.q_split <= full.q_split && sp.part_bytes <= full.part_bytes,
                    "a device of %d CUs asks for more than the workspace query grants (B%d N%d Sq%d Sk%d D%d)", n_cu, B, N, Sq, Sk, D);
              if (sp.q_split > 1) {
                CHECK(sp.q_split * n_wg <= (n_cu > 256 ? 256 : n_cu), "split grid %lld exceeds the CUs", sp.q_split * n_wg);
                CHECK(((Sq + 63) / 64) / sp.q_split >= 8, "a slice has fewer than 512 query rows");
                CHECK(sp.part_bytes == (size_t)sp.q_split * n_wg * 8 * ngk * db * 4096, "part_bytes");
              } else {
                CHECK(sp.part_bytes == 0, "no split but %zu bytes", sp.part_bytes);
              }
            }
  // the cross-attention shape the split exists for, and the benchmark shape that must not split
  CHECK(dkdv_split(2, 16, 4096, 77, 40).q_split == 8, "B2 N16 Sq4096 Sk77 D40 -> %d", dkdv_split(2, 16, 4096, 77, 40).q_split);
  CHECK(dkdv_split(4, 16, 2048, 2048, 128).q_split == 1, "the benchmark shape splits");
}

// key slices of the forward kernel: any number that fits one round of workgroups, none of them empty, room as stated;
// query slices of the dK/dV kernel: no more room than there is
static void test_slice_plans() {
  for (int BH : {1, 3, 5, 7, 24, 40, 56, 200})
    for (int Sq : {1, 65, 300, 513, 1611, 4096})
      for (int Sk : {1, 77, 130, 1000, 8197, 131072})
        for (int D : {40, 64, 80, 128, 160, 256})
          for (int n_cu : {32, 256})
            for (bool tri : {false, true}) {
              const FwdPlan f = fwd_plan(1, BH, Sq, Sk, D, false, tri, true, n_cu);
              const int rows = head_dim_class(D) > 160 ? 128 : 256 / f.kg, tiles = ((tri && Sq < Sk ? Sq : Sk) + 127) / 128;
              CHECK(f.part_bytes == fwd_part_bytes(1, BH, Sq, D, f.kg, f.kv_split), "part_bytes");
              if (f.kv_split > 1) {
                const int walk = (tiles + f.kv_split - 1) / f.kv_split;
                CHECK((long long)f.kv_split * BH * ((Sq + rows - 1) / rows) <= n_cu, "%d slices do not fit", f.kv_split);
                CHECK((f.kv_split - 1) * walk < tiles, "an empty slice: %d of %d tiles", f.kv_split, tiles);
              }
              CHECK(fwd_plan(1, BH, Sq, Sk, D, false, tri, false, n_cu).kv_split == 1, "a split without room");
              for (size_t room : {(size_t)0, (size_t)1 << 22, SIZE_MAX}) {
                const DkdvPlan p = dkdv_plan(1, BH, Sq, Sk, D, tri, room, n_cu);
                CHECK(p.part_bytes <= room && p.part_bytes == dkdv_part_bytes(1, BH, Sk, D, p.ngk, p.q_split), "part_bytes");
                CHECK(p.q_split == 1 || (long long)p.q_split * BH * ((Sk + 128 * p.ngk - 1) / (128 * p.ngk)) <= (tri ? 2 : 1) * n_cu,
                      "%d slices do not fit", p.q_split);
              }
            }
  CHECK(fwd_plan(1, 3, 300, 60000, 128, false, false, true).kv_split == 28, "9 workgroups, 256 CUs");
}

// the longest walk of a 128-row block, counted key block by key block
static void test_visible_row_keys() {
  for (int Sq : {1, 128, 129, 1000, 8192})
    for (int Sk : {1, 77, 128, 1000, 8192, 8200})
      for (int prev : {0, 1, 3, 65536})
        for (int next : {0, 1, 5, 65536, 0x7fffffff})
          for (int prefix : {0, 128, 1024, 4096}) {
            int most = 0;
            for (int qb = 0; qb < (Sq + 127) / 128; qb++) {
              int lo = Sk, hi = 0;
              for (int j = 0; j < Sk; j++) {
                if (j / 128 > (long long)qb + next || qb > (long long)j / 128 + prev) continue;
                if (prefix && j >= (qb * 128 / prefix + 1) * prefix) continue;
                if (j < lo) lo = j;
                hi = j + 1;
              }
              if (hi - lo > most) most = hi - lo;
            }
            const int keys = visible_row_keys(Sq, Sk, prev, next, prefix);
            CHECK(keys >= most && keys <= Sk, "Sq %d Sk %d band %d/%d prefix %d: %d keys, %d visible", Sq, Sk, prev, next, prefix, keys, most);
            if (!prefix && prev == 65536 && next == 65536) CHECK(keys == Sk, "no band");
          }
  CHECK(visible_row_keys(8192, 8192, 1, 1, 0) == 384 && visible_row_keys(8192, 8192, 2, 0, 0) == 384, "three key blocks");
  CHECK(visible_row_keys(1000, 9000, 65536, 65536, 512) == 1024, "two groups of rows");
  // below the diagonal on long walks, up to twice as many units as CUs end together: no finer ones
  for (int S : {3500, 4096}) CHECK(dkdv_plan(1, 32, S, S, 64, true, SIZE_MAX).ngk == 2, "S%d", S);
  CHECK(dkdv_plan(1, 32, 3000, 3000, 64, true, SIZE_MAX).ngk == 1 && dkdv_plan(1, 80, 1500, 1500, 64, true, SIZE_MAX).ngk == 1, "finer units");
  CHECK(dkdv_plan(1, 64, 4096, 4096, 64, true, SIZE_MAX).ngk == 1 && dkdv_plan(1, 16, 2048, 2048, 128, true, SIZE_MAX).q_split == 1, "finer units");
  // the dK/dV units of a band: as few as fill the CUs where the band is wide, finer ones where it is narrow
  CHECK(dkdv_plan(2, 16, 2048, 2048, 128, false, SIZE_MAX, 256, 8, 0).ngk == 2, "256 workgroups of a wide band");
  CHECK(dkdv_plan(3, 16, 1500, 1500, 80, false, SIZE_MAX, 256, 5, 0).ngk == 2, "288 workgroups, those at the end shorter");
  CHECK(dkdv_plan(4, 16, 4096, 4096, 64, false, SIZE_MAX, 256, 1, 0).ngk == 1, "a narrow band");
  // a band of three key blocks is one launch, whatever the length; a wide one is cut, by what its rows see
  CHECK(fwd_plan(1, 1, 8192, 8192, 64, false, false, true, 256, visible_row_keys(8192, 8192, 1, 1, 0)).kv_split == 1, "a narrow band is cut");
  CHECK(fwd_plan(1, 1, 256, 131072, 128, false, false, true, 256, visible_row_keys(256, 131072, 0, 2, 0)).kv_split == 1, "few keys are cut");
  CHECK(fwd_plan(1, 1, 256, 131072, 128, false, false, true, 256, visible_row_keys(256, 131072, 65536, 200, 0)).kv_split > 8, "a wide band is not cut");
}

// every (slice, workgroup) once; shared: the row tiles of a head and slice next to each other on one XCD (but where its share
// ends); plain: on one XCD where the heads are a multiple of 8, which is why such launches do not share
static void test_split_map() {
  for (bool share : {true, false})
    for (int BH : {1, 3, 8, 40, 64, 100, 128})
      for (int n_tiles : {1, 2, 3, 5})
        for (int split : {2, 3, 7, 16, 128}) {
          if (BH == 128 && n_tiles > 1) continue;                                        // (such a launch is not cut)
          const int n = BH * n_tiles * split;
          std::vector<int> seen(n, -1);
          int apart = 0, other_xcd = 0;
          for (int id = 0; id < n; id++) {
            int slice = -1, wg = -1;
            split_map(id, BH, n_tiles, split, share, slice, wg);
            const bool in = slice >= 0 && slice < split && wg >= 0 && wg < BH * n_tiles;
            CHECK(in, "BH %d tiles %d split %d id %d: slice %d wg %d", BH, n_tiles, split, id, slice, wg);
            if (!in) continue;
            CHECK(seen[slice * BH * n_tiles + wg] < 0, "BH %d tiles %d split %d id %d: twice", BH, n_tiles, split, id);
            seen[slice * BH * n_tiles + wg] = id;
          }
          for (int slice = 0; slice < split && n_tiles > 1; slice++)
            for (int bh = 0; bh < BH; bh++)
              for (int t = 1; t < n_tiles; t++) {
                const int id = seen[slice * BH * n_tiles + t * BH + bh], before = seen[slice * BH * n_tiles + (t - 1) * BH + bh];
                apart += id != before + 8;
                other_xcd += id % 8 != before % 8;
              }
          if (share) CHECK(apart <= 8, "BH %d tiles %d split %d: %d neighbours apart", BH, n_tiles, split, apart);
          else CHECK((other_xcd == 0) == (BH % 8 == 0 || n_tiles == 1), "BH %d tiles %d split %d: %d on other XCDs", BH, n_tiles, split, other_xcd);
        }
  CHECK(split_shares(1, 131072, 128) && split_shares(2, 100000, 64) && split_shares(1, 110000, 64) && split_shares(12, 9200, 64), "more than the L2s hold");
  CHECK(!split_shares(1, 109000, 64) && !split_shares(3, 16000, 128) && !split_shares(8, 131072, 128) && !split_shares(64, 8192, 128), "nothing to gain");
}

// the mean of what the rows see, against a count
static void test_pipelined_walks() {
  for (int Sq : {1, 100, 256, 1000, 3000})
    for (int Sk : {1, 77, 1024, 5000}) {
      long long all = 0;
      for (int i = 0; i < Sq; i++) all += i + 1 < Sk ? i + 1 : Sk;
      const double mean = (double)all / Sq;
      const long long got = mean_row_keys(Sq, Sk, true);
      CHECK(got >= mean - 2 && got <= mean + 2, "Sq %d Sk %d: %lld, %.1f", Sq, Sk, got, mean);
      CHECK(mean_row_keys(Sq, Sk, false) == Sk, "all rows see all keys");
    }
  CHECK(!pipelined_pays(4096, 1023, false) && pipelined_pays(256, 1024, false), "short and long walks");
  CHECK(!pipelined_pays(2046, 2046, true) && pipelined_pays(2048, 2048, true) && !pipelined_pays(256, 8192, true), "causal walks");
  CHECK(first_tile_late(257, 1, 128, 128) && !first_tile_late(256, 1, 128, 128) && !first_tile_late(512, 2, 128, 128) && !first_tile_late(512, 1, 129, 128), "one tile");
  CHECK(!pipelined_pays(8192, visible_row_keys(8192, 8192, 3, 3, 0), false) && pipelined_pays(8192, visible_row_keys(8192, 8192, 4, 4, 0), false), "bands");
}

// 256-key tiles of small grids: as many tiles of either length as the longest walk touches, wherever it starts
static void test_long_tiles() {
  for (int seen = 1; seen <= 3000; seen += seen % 128 == 0 || seen % 128 == 127 ? 1 : 126)
    for (int moving = 0; moving < 2; moving++) {
      int most = 0;                                        // of the 256-key tiles that hold `blocks` blocks from any one on
      const int blocks = (seen + 127) / 128;
      for (int first = 0; first < (moving ? 2 : 1); first++) most = std::max(most, (first + blocks - 1) / 2 + 1);
      CHECK(long_tiles_pay(4, 512, 4096, 64, seen, moving) == (blocks > 1.65 * most), "%d keys, moving %d", seen, moving);
    }
  for (int Sk : {129, 256, 400, 512, 600, 2000}) CHECK(long_tiles_pay(16, 512, Sk, 64, Sk, false), "Sk %d", Sk);
  for (int Sk : {1, 128, 257, 384}) CHECK(!long_tiles_pay(16, 512, Sk, 64, Sk, false), "Sk %d", Sk);
  CHECK(!long_tiles_pay(257, 64, 500, 40, 500, false) && long_tiles_pay(256, 64, 500, 40, 500, false), "one round");
  CHECK(!long_tiles_pay(250, 64, 600, 64, 600, false) && long_tiles_pay(250, 64, 512, 64, 512, false) && long_tiles_pay(250, 64, 1024, 40, 1024, false), "keys from memory");
}

// the largest offset of a tile, as TileDma keeps it: (r * stride + 8 chunk) * 2 bytes in 32 bits
static void test_tile_offsets() {
  for (int rows : {64, 128, 256})
    for (int64_t stride : {int64_t(64), int64_t(1) << 23, int64_t(9) << 20, int64_t(1) << 24, (int64_t(1) << 24) + (1 << 20), kBwdRowStrideEnd - 8, kBwdRowStrideEnd,
                           int64_t(35) << 20, int64_t(1) << 31, int64_t(1) << 40}) {
      const int64_t most = ((rows - 1) * stride + 256) * 2;
      CHECK(tile_offsets_fit(stride, rows) == (most <= 0xffffffffll), "%d rows, stride %lld", rows, (long long)stride);
    }
  CHECK(tile_offsets_fit(kBwdRowStrideEnd - 8, 64) && !tile_offsets_fit(kBwdRowStrideEnd, 64), "where the backward's strides end");
  CHECK(tile_offsets_fit(16909312, 128) && !tile_offsets_fit(16909320, 128), "where the forward's strides end");
  CHECK(!tile_offsets_fit(int64_t(9) << 20, 256) && tile_offsets_fit(int64_t(9) << 20, 128), "256-key tiles reach half as far");
}

static void test_div_small() {
  for (int n = 1; n <= 32; n++)
    for (int idx = 0; idx < 1024; idx++) CHECK(div_small(idx, recip16(n)) == idx / n, "div_small(%d, %d)", idx, n);
}

// a workgroup's base and a lane's 32-bit offset reach the entry of every one of its keys, also where 16 bytes a key pass 4 GB
static void test_keep_columns() {
  for (int Sk : {1, 200, 4096, (1 << 28) + 200, 0x7fffff00})
    for (int k0 : {0, 128, Sk / 256 * 256, (Sk - 1) / 128 * 128})
      for (int t : {0, 1, 127, 255}) {
        if (k0 >= Sk) continue;
        const int dk = t < Sk - 1 - k0 ? t : Sk - 1 - k0, key = k0 + dk;
        const int64_t want = ((((int64_t)5 * 3 + 2) * Sk + key) * 4 + 1) * 4;          // (head 5, block 2 of 3, word 1)
        const uint32_t off = keep_col_offset(dk, 1);
        CHECK(keep_col_entry(5, 3, 2, Sk, k0) * 4 + off == want && off < 4096, "Sk %d k0 %d key %d", Sk, k0, key);
      }
}

int main() {
  test_wg_map();
  test_swizzle_rows<64>();
  test_swizzle_rows<128>();
  test_swizzle_rows<256>();
  test_tr_hi<64>();
  test_tr_hi<128>();
  test_tr_hi<256>();
  test_head_dim_class();
  test_dkdv_split();
  test_slice_plans();
  test_visible_row_keys();
  test_keep_columns();
  test_split_map();
  test_tile_offsets();
  test_pipelined_walks();
  test_long_tiles();
  test_div_small();
  if (failures) printf("%d checks failed\n", failures);
  else printf("index math: all checks passed\n");
  return failures > 255 ? 255 : failures;
}
