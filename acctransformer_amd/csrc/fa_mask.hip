// Block classification of a dense attention mask (uint8, or the I/O dtype as the reference passes it;
// nonzero = masked either way).
//
// The reference adds -10000 to masked scores (attention.py:357-371 of the
// reference's flash_attention ops) instead of removing them.  A 128x128 block
// whose entries are all masked therefore contributes exp(-10000 + ...) = 0 in
// fp32 to every row that has at least one unmasked visible key elsewhere, and
// can be skipped without changing a bit of the result; a block with no masked
// entry needs no mask loads.  This pre-pass finds both kinds so the attention
// kernels touch the mask only on mixed blocks.  A diagonal block (same 128 rows and keys) whose entries
// are exactly "masked iff the key comes after the query" - every diagonal block of a causal mask given
// as a tensor, with or without padding elsewhere - gets a class of its own: the kernels then compare
// indices there, as they do for the causal mask kind, instead of loading mask bytes.
#include "fa_common.hpp"
#include "fa_launch.hpp"

namespace acct {

// ONE launch leaves the block classes and, for the dK/dV kernel, the column bitmaps of the mixed blocks (every
// launch costs a few microseconds of a step that takes a few hundred).  One workgroup of 256 threads per (mask
// batch, q block, key block) inside the band, so that the work spreads over the chip whatever the shape (a
// [1, 2048, 2048] mask has 16 row blocks but 256 blocks).  Thread t owns 64 consecutive elements of row t % 128
// (half t / 128 of the block's 128 columns), four or eight 16-byte loads at whatever alignment the rows have (a
// sequence length that is no multiple of 16 shifts every row; such loads touch one cache line more, no more
// instructions), as a 64-bit "nonzero" mask.
//
// A wholly masked block may be skipped only if every row of its q block sees an unmasked key somewhere (see the
// top of the file).  A workgroup cannot see the other blocks of its row block's band, so it checks a sufficient
// condition on two of them that it reads itself: every row has an unmasked key in the first block of the band
// or in the diagonal block.  That holds for causal, banded, prefix and document masks (the diagonal entry is
// visible) and for key padding (the first keys are); where it fails although the rows do see keys elsewhere,
// the block is classed 'apply' instead of 'skip', which gives the same results bit for bit, only slower.
template <int ES>
__global__ void __launch_bounds__(256) fa_mask_prepass_kernel(const FaArgs a, uint8_t* flags, uint8_t* tails, uint32_t* colbits) {
  __shared__ unsigned long long s_bits[128][2];         // nonzero bits of the block: [row][column half]
  __shared__ unsigned long long s_seen[2];              // rows (bit = row % 64) with an unmasked key in the blocks probed
  __shared__ int s_lead[2];                             // unmasked leading columns of the block's first row, per column half
  const int kvb = blockIdx.x % a.Tc, qb = (blockIdx.x / a.Tc) % a.Tr, mb = blockIdx.x / (a.Tc * a.Tr);
  const int tid = threadIdx.x;
  int lo = max(0, qb - a.prev_blk), hi = min(a.Tc - 1, qb + a.next_blk);
  if (a.row_prefix) hi = min(hi, ((qb * 128 / a.row_prefix + 1) * a.row_prefix - 1) / 128);
  const int64_t blk = ((int64_t)mb * a.Tr + qb) * a.Tc + kvb;
  if (kvb < lo || kvb > hi) {                           // outside the band: never visited
    if (tid == 0) { flags[blk] = kBlkClean; tails[blk] = 0; }
    return;
  }
  const int rib = tid & 127, half = tid >> 7, row = qb * 128 + rib, c0 = half * 64;
  const uint8_t* mrow = a.mask + ((int64_t)mb * a.mask_sb + (int64_t)min(row, a.Sq - 1) * a.Sk) * ES;
  // this thread's 64 elements of key block kb: nz = nonzero bits, valid = bits of the elements that exist
  auto scan = [&](int kb, unsigned long long& nz, unsigned long long& valid) {
    nz = 0; valid = 0;
    if (row >= a.Sq) return;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int kv = kb * 128 + c0 + 16 * i;
      if (kv >= a.Sk) continue;
      uint32_t bits = 0;                                // bit e: element e of these 16 is nonzero
      if (kv + 16 <= a.Sk) {
#pragma unroll
        for (int h = 0; h < ES; h++) {
          const u32x4 v = load_any<u32x4, ES>(mrow + (int64_t)kv * ES + 16 * h);
#pragma unroll
          for (int w = 0; w < 4; w++) {
            if (ES == 1) {
#pragma unroll
              for (int e = 0; e < 4; e++) bits |= (((v[w] >> (8 * e)) & 0xffu) != 0 ? 1u : 0u) << (4 * w + e);
            } else {
              // 2-byte floating-point elements: the sign of a zero does not count
              bits |= (((v[w] & 0x7fffu) != 0 ? 1u : 0u) | (((v[w] >> 16) & 0x7fffu) != 0 ? 2u : 0u)) << (8 * h + 2 * w);
            }
          }
        }
        valid |= 0xffffull << (16 * i);
      } else {                                          // the row ends inside this piece
        for (int e = 0; e < a.Sk - kv; e++) bits |= (elem_nonzero<ES>(mrow, kv + e) ? 1u : 0u) << e;
        valid |= ((1ull << (a.Sk - kv)) - 1ull) << (16 * i);
      }
      nz |= (unsigned long long)bits << (16 * i);
    }
  };
  unsigned long long nz, valid;
  scan(kvb, nz, valid);
  // the causal pattern on the diagonal block: column c0 + e is masked iff it comes after row rib
  const int d = rib - c0;                               // columns above bit d are "after the row"
  const unsigned long long tri = d < 0 ? ~0ull : (d >= 63 ? 0ull : (~0ull << (d + 1)));
  const bool on_diag = kvb == qb;
  const int any_m = __syncthreads_or(nz != 0), any_u = __syncthreads_or((~nz & valid) != 0);
  const int bad = __syncthreads_or(on_diag && ((nz ^ tri) & valid) != 0);
  uint8_t cls = !any_m ? kBlkClean : (any_u ? ((on_diag && !bad) ? kBlkTriu : kBlkApply) : kBlkSkip);
  if (cls == kBlkSkip) {                                // (uniform: the whole workgroup takes the branch)
    if (tid < 2) s_seen[tid] = 0;
    __syncthreads();
    const int probe[2] = {lo, (qb >= lo && qb <= hi && qb != lo) ? qb : -1};
#pragma unroll
    for (int k = 0; k < 2; k++)
      if (probe[k] >= 0 && probe[k] != kvb) {
        unsigned long long pnz, pvalid;
        scan(probe[k], pnz, pvalid);
        const unsigned long long seen = __ballot((~pnz & pvalid) != 0);
        if ((tid & 63) == 0 && seen) atomicOr(&s_seen[(tid >> 6) & 1], seen);
      }
    __syncthreads();
    const int nrow = min(128, a.Sq - qb * 128);         // rows past Sq do not count
    bool ok = true;
#pragma unroll
    for (int w = 0; w < 2; w++) {
      const int n = min(64, max(0, nrow - 64 * w));
      const unsigned long long need = n >= 64 ? ~0ull : ((1ull << n) - 1ull);
      ok = ok && (s_seen[w] & need) == need;
    }
    if (!ok) cls = kBlkApply;
  }
  // A mixed block in which every row masks exactly the columns from the t-th on (1 <= t <= 127; key padding that
  // ends inside the block): the forward and dQ kernels compare key indices with t there instead of loading mask
  // bytes.  t is taken from the block's first row (which always exists) and checked against every row.
  int tail = 0;
  if (cls == kBlkApply) {                               // (uniform)
    if (rib == 0) s_lead[half] = nz ? __builtin_ctzll(nz) : 64;
    __syncthreads();
    const int t = s_lead[0] < 64 ? s_lead[0] : 64 + s_lead[1];
    const int rel = t - c0;                             // this thread's columns from bit `rel` on are masked
    const unsigned long long want = rel <= 0 ? ~0ull : (rel >= 64 ? 0ull : (~0ull << rel));
    const int differs = __syncthreads_or(row < a.Sq && ((nz ^ want) & valid) != 0);
    if (!differs && t >= 1 && t <= 127) tail = t;
  }
  if (tid == 0) { flags[blk] = cls; tails[blk] = (uint8_t)tail; }
  if (cls == kBlkApply && colbits) {
    // the block packed by key column: 128 bits per key, bit r = mask[128 qb + r][key]
    s_bits[rib][half] = nz;
    __syncthreads();
    const int col = tid & 127, kv = kvb * 128 + col;
    if (kv < a.Sk) {
      const ACCT_LDS uint32_t* sb = (const ACCT_LDS uint32_t*)&s_bits[0][0] + (col >> 5);   // the 32-bit piece that holds the column
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int i = 2 * half + j;
        uint32_t w = 0;
#pragma unroll 8
        for (int r = 0; r < 32; r++) w |= ((sb[(32 * i + r) * 4] >> (col & 31)) & 1u) << r;
        colbits[(((int64_t)mb * a.Tr + qb) * a.Sk + kv) * 4 + i] = w;
      }
    }
  }
}

// The compact 128x128 tile that is applied on diagonal blocks, packed by key column for the dK/dV kernel, whose lanes
// own key columns: out[key][4], bit r of the 128-bit entry = tile[r][key]
template <int ES>
__global__ void __launch_bounds__(128) fa_mask_tilebits_kernel(const uint8_t* tile, uint32_t* out) {
  uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll 8
    for (int r = 0; r < 32; r++)
      if (elem_nonzero<ES>(tile, (32 * i + r) * 128 + threadIdx.x)) w[i] |= 1u << r;
  u32x4 v = {w[0], w[1], w[2], w[3]};
  *reinterpret_cast<u32x4*>(out + threadIdx.x * 4) = v;
}

hipError_t launch_mask_tilebits(const FaArgs& a, uint32_t* out, hipStream_t st) {
  if (a.mask_es == 2) hipLaunchKernelGGL(fa_mask_tilebits_kernel<2>, dim3(1), dim3(128), 0, st, a.mask, out);
  else hipLaunchKernelGGL(fa_mask_tilebits_kernel<1>, dim3(1), dim3(128), 0, st, a.mask, out);
  return hipGetLastError();
}

// Key blocks whose keep bits no attention kernel reads: those that the attention mask's pre-pass classed 'skip', and
// those that the band, the causal index compare or the row prefix leaves out for every row of the q block.  (Those only
// with `drop_visible`: calls with another band may share a lent buffer of keep bits, unless the caller rules it out.)
// `flags`: the class row of the q block, or null.
ACCT_DEV bool keep_bits_unread(const FaArgs& a, const uint8_t* flags, int qb, int kvb) {
  if (flags && flags[kvb] == kBlkSkip) return true;
  if (!a.drop_visible) return false;
  return kvb - a.next_blk > qb || qb > kvb + a.prev_blk || (a.mask_kind == kMaskCausal && kvb > qb) ||
         (a.row_prefix && kvb * 128 >= (qb * 128 / a.row_prefix + 1) * a.row_prefix);
}

// Both dropout pre-passes below work in units of ONE WAVE per (batch*head, 128 query rows, 128 keys), a block that is
// either left out as a whole or needed; a workgroup's four waves take neighbouring key blocks.  A lane holds the keep
// bits of a piece of the block, puts its bits of every row and its words of every key column into a wave-private LDS
// image of the block's two outputs, and the wave stores the image: whole 16-byte column entries, consecutive lanes
// consecutive entries, and 16-byte row pieces.  (Written straight from the lanes, an entry would be four or eight
// stores.)  One spare 16-byte entry after every sixteen keeps the lanes' pieces on different banks.
constexpr int kKeepImage = 128 + 8;                      // 16-byte entries of one output of a block
struct KeepBlock {
  int kvb, qb, bh, lane;
  ACCT_LDS char* row;                                    // [row][16 bytes]: bit k = keep[row][128 kvb + k]
  ACCT_LDS char* col;                                    // [key][16 bytes]: bit r = keep[128 qb + r][key]
  static ACCT_DEV int at(int i) { return (i + (i >> 4)) * 16; }
  // false: nothing to do for this wave
  ACCT_DEV bool init(const FaArgs& a, ACCT_LDS char* lds, int blk) {
    const int wave = threadIdx.x >> 6, nspan = (a.Tc + 3) / 4;
    lane = threadIdx.x & 63;
    kvb = __builtin_amdgcn_readfirstlane(4 * (blk % nspan) + wave);
    qb = (blk / nspan) % a.Tr;
    bh = blk / (nspan * a.Tr);
    row = lds + wave * (2 * kKeepImage * 16);
    col = row + kKeepImage * 16;
    if (kvb >= a.Tc) return false;
    return !keep_bits_unread(a, a.blkflags ? a.blkflags + ((int64_t)(a.mask_sb ? bh / a.N : 0) * a.Tr + qb) * a.Tc : nullptr, qb, kvb);
  }
  ACCT_DEV void store(const FaArgs& a, uint32_t* rowbits, uint32_t* colbits) const {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (a wave's LDS operations complete in order: its lanes see each other's)
#pragma unroll
    for (int m = 0; m < 2; m++) {
      const int i = lane + 64 * m, r = qb * 128 + i, key = kvb * 128 + i;
      if (rowbits && r < a.Sq) {
        const u32x4 w = *reinterpret_cast<const ACCT_LDS u32x4*>(row + at(i));
        // (an even number of words per row: 8-byte pieces, the second half of the last block may lie past the row)
        uint32_t* out = rowbits + ((int64_t)bh * a.Sq + r) * a.droprow_w + 4 * kvb;
        const u32x2 w0 = {w[0], w[1]}, w1 = {w[2], w[3]};
        *reinterpret_cast<u32x2*>(out) = w0;
        if (4 * kvb + 2 < a.droprow_w) *reinterpret_cast<u32x2*>(out + 2) = w1;
      }
      if (colbits && key < a.Sk)
        *reinterpret_cast<u32x4*>(colbits + (((int64_t)bh * a.Tr + qb) * a.Sk + key) * 4) = *reinterpret_cast<const ACCT_LDS u32x4*>(col + at(i));
    }
  }
};

// 8 x 8 bit transposes of all four bytes of x[0..7] at once: bit k of byte b of x[j] <-> bit j of byte b of x[k]
ACCT_DEV void transpose_bytes8(uint32_t (&x)[8]) {
  uint32_t mask = 0x0f0f0f0fu;
#pragma unroll
  for (int sft = 4; sft >= 1; sft >>= 1) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (k & sft) continue;
      const uint32_t t = ((x[k] >> sft) ^ x[k + sft]) & mask;
      x[k + sft] ^= t;
      x[k] ^= t << sft;
    }
    mask ^= mask << (sft >> 1);
  }
}
// the column words of sixteen keys x sixteen rows: x[j] holds rows j (low half) and j + 8 (high half), bit = key;
// afterwards keys j and j + 8, bit = row
ACCT_DEV void transpose_16x16(uint32_t (&x)[8]) {
#pragma unroll
  for (int j = 0; j < 8; j++) x[j] = __builtin_amdgcn_perm(x[j], x[j], 0x03010200u);   // the off-diagonal bytes change places
  transpose_bytes8(x);
}

// sixteen bytes at any address that nothing reads again
typedef u32x4 u32x4_any __attribute__((aligned(1)));
ACCT_DEV u32x4 load_once(const uint8_t* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p)); }

// Dropout mask (uint8 {0,1}, or the reference's {0, 1/keep_prob} in the I/O dtype; nonzero = keep) packed into keep bits, by query row for the kernels whose lanes own
// query rows (forward, dQ) and by key column for the dK/dV kernel.
//   rowbits [B*N*Sq, 2*ceil(Sk/64)] 32-bit: bit k of word w = keep[row][32w + k];
//   colbits [B*N, Tr, Sk, 4] 32-bit: bit r of the 128-bit entry = keep[128*qb + r][key].
// Bound by the mask bytes it reads.  A wave's load instruction reads the block's 128 or 256 bytes of eight or four
// rows, sixteen such loads in flight, at any alignment (a key count that is no multiple of 16 shifts every row).
// Blocks whose bits no kernel reads are not loaded.  Before, a wave walked 32 rows of 1024 keys: hidden blocks then
// left lanes idle but saved no instruction, and those bound it: B4 N8 S4096 causal, 2-byte mask (half of 1.07 GB
// is needed) 274.7 -> 185.1 us.  Neighbouring blocks share the lines of the row words and of each mask row's pages:
// each XCD takes one contiguous eighth of them, and the mask, read once, does not displace anything in the caches:
// 155.5 us with the first alone, 175.1 with the second alone, 142.3 = 4.2 TB/s with both; S3001, 3 x 8 heads 83.9 ->
// 82 to 86, S1024 12.6 -> 11.1 to 11.8 over the runs seen.  (The Philox kernel below reads nothing, and an eighth of its blocks each evens out less
// well: 46.5 -> 48.8 on a padded batch, so it takes them in order.)
template <int ES>
__global__ void __launch_bounds__(256) fa_drop_bits_kernel(const FaArgs a, uint32_t* rowbits, uint32_t* colbits) {
  __shared__ __attribute__((aligned(16))) char s_img[4 * 2 * kKeepImage * 16];
  KeepBlock kb;
  if (!kb.init(a, (ACCT_LDS char*)s_img, xcd_span(blockIdx.x, gridDim.x))) return;
  constexpr int KH = 16 / ES, LPR = 128 / KH, NR = 2 * LPR;   // keys per load; lanes per row; rows of a lane (16 for bytes, 32 for 2-byte elements)
  const int c = kb.lane % LPR, R = kb.lane / LPR;
  const int row0 = kb.qb * 128 + NR * R, kv = kb.kvb * 128 + KH * c;
  const int nrow = min(NR, a.Sq - row0);
  const uint8_t* p = a.drop + (((int64_t)kb.bh * a.Sq + row0) * a.Sk + kv) * ES;
  uint32_t cw[8];                                        // bytes: rows j, j + 8 in the halves; 2-byte: rows j, j + 8, j + 16, j + 24 in the bytes
#pragma unroll
  for (int j = 0; j < 8; j++) cw[j] = 0u;
  auto take = [&](int j, uint32_t nz) {                  // nz: bit e = key e of this lane is kept in its row j
    ACCT_LDS char* out = kb.row + KeepBlock::at(NR * R + j);
    if (ES == 1) {
      *reinterpret_cast<ACCT_LDS uint16_t*>(out + 2 * c) = (uint16_t)nz;
      cw[j & 7] |= nz << (16 * (j >> 3));
    } else {
      *reinterpret_cast<ACCT_LDS uint8_t*>(out + c) = (uint8_t)nz;
      cw[j & 7] |= nz << (8 * (j >> 3));
    }
  };
  auto pack = [&](const u32x4& v) {
    uint32_t nz = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      if (ES == 1) {
        // bit 7 of byte e: nonzero (no carry leaves a byte); the dot product with 1 2 4 8 (16 32 64 128) gathers the bits
        const uint32_t y = (((v[w] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v[w]) & 0x80808080u;
        nz += __builtin_amdgcn_udot4(y, w & 1 ? 0x80402010u : 0x08040201u, 0u, false) << (8 * (w >> 1));
      } else {
        // 2-byte floating-point elements: nonzero apart from the sign bit
        const uint32_t y = ((v[w] & 0x7fff7fffu) + 0x7fff7fffu) & 0x80008000u;
        nz |= (y >> (15 - 2 * w)) | (y >> (30 - 2 * w));
      }
    }
    return ES == 1 ? nz >> 7 : nz & 0xffu;
  };
  if (kb.qb * 128 + 128 <= a.Sq && kb.kvb * 128 + 128 <= a.Sk) {   // (wave-uniform: no lane tests anything)
#pragma unroll
    for (int r0 = 0; r0 < NR; r0 += 16) {
      u32x4 v[16];
#pragma unroll
      for (int j = 0; j < 16; j++) {
        v[j] = load_once(p);
        p += (int64_t)a.Sk * ES;
      }
#pragma unroll
      for (int j = 0; j < 16; j++) take(r0 + j, pack(v[j]));
    }
  } else {
    const bool whole = kv + KH <= a.Sk;
#pragma unroll
    for (int j = 0; j < NR; j++) {
      uint32_t nz = 0;
      if (j < nrow) {
        if (whole) nz = pack(load_any<u32x4, ES>(p));
        else                                             // the row ends inside (or before) this lane's piece
          for (int e = 0; e < a.Sk - kv; e++) nz |= (elem_nonzero<ES>(p, e) ? 1u : 0u) << e;
      }
      take(j, nz);
      p += (int64_t)a.Sk * ES;
    }
  }
  if (ES == 1) transpose_16x16(cw);
  else transpose_bytes8(cw);
#pragma unroll
  for (int t = 0; t < KH; t++) {
    ACCT_LDS char* out = kb.col + KeepBlock::at(KH * c + t);
    if (ES == 1) *reinterpret_cast<ACCT_LDS uint16_t*>(out + 2 * R) = (uint16_t)(cw[t & 7] >> (16 * (t >> 3)));
    else *reinterpret_cast<ACCT_LDS uint32_t*>(out + 4 * R) = cw[t & 7];
  }
  kb.store(a, rowbits, colbits);
}

// The same bitmaps for counter-based dropout: nothing is read, the keep decisions come from Philox4x32-10.
// One call yields the 16 bytes of one (query row, 32-key group M, half g): keys 32M + 8u + 4g + e for
// u = 0..3, e = 0..3 -- the keys one lane of the attention kernels owns in a 32-key group, so a kernel
// could also draw them in place.
// Bound by vector instructions: the ten rounds' twenty 32 x 32 -> 64-bit products, a quarter-rate instruction each,
// are more than half of them.  Lane 8R + 2M + g draws rows 16R .. +15 of (M, g).  The sixteen byte comparisons of a
// call are done on whole words, four dot products gather their outcomes into sixteen adjacent bits, and the column
// words come from a bit-matrix transpose in registers.
// Padded batch B16 N16 S1024, 69 % of the blocks visible: 73.6 -> 48.0 us (a wave that walked 32 rows of all keys
// drew the hidden ones too, and compared and shifted key by key).
__global__ void __launch_bounds__(256) fa_drop_philox_kernel(const FaArgs a, uint32_t* rowbits, uint32_t* colbits) {
  __shared__ __attribute__((aligned(16))) char s_img[4 * 2 * kKeepImage * 16];
  KeepBlock kb;
  if (!kb.init(a, (ACCT_LDS char*)s_img, blockIdx.x)) return;
  const int g = kb.lane & 1, M = (kb.lane >> 1) & 3, R = kb.lane >> 3;
  const int row0 = kb.qb * 128 + 16 * R;
  // byte < thr on four bytes at once: with bit 7 set aside the difference stays inside its byte, and its bit 7 joins
  // the two sevenths bits: not (x & z) for thr >= 128, not (x | z) below -- the majority with a constant.
  const uint32_t thr7 = (a.philox_thr & 0x7fu) * 0x01010101u, low = a.philox_thr & 0x80u ? 0u : ~0u;
  const uint32_t all = a.philox_thr >= 256u ? 0x80808080u : 0u;
  uint32_t cw[8];                                       // rows j (low half) and j + 8 (high half), bit 4u + e
#pragma unroll
  for (int j = 0; j < 8; j++) cw[j] = 0u;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int row = row0 + r;
    uint32_t v[4];
    philox4x32_10((uint32_t)row, (uint32_t)(2 * (4 * kb.kvb + M) + g), (uint32_t)kb.bh, a.philox_offset, a.philox_k0, a.philox_k1, v);
    uint32_t y[4];                                      // bit 7 of byte e: kept
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const uint32_t z = (v[u] | 0x80808080u) - thr7;
      y[u] = (~((v[u] & z) | ((v[u] | z) & low)) & 0x80808080u) | all;
    }
    // byte weights 1 2 4 8 and 16 32 64 128: 128 times the eight bits of two words
    const uint32_t b01 = __builtin_amdgcn_udot4(y[1], 0x80402010u, __builtin_amdgcn_udot4(y[0], 0x08040201u, 0u, false), false);
    const uint32_t b23 = __builtin_amdgcn_udot4(y[3], 0x80402010u, __builtin_amdgcn_udot4(y[2], 0x08040201u, 0u, false), false);
    uint32_t bits = (b01 >> 7) | (b23 << 1);
    uint32_t x = (bits | (bits << 8)) & 0x00ff00ffu;    // nibble u to byte u
    x = ((x | (x << 4)) & 0x0f0f0f0fu) << (4 * g);
    x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xf, 0xf, true);    // lane ^ 1: the other half
    if (g == 0) *reinterpret_cast<ACCT_LDS uint32_t*>(kb.row + KeepBlock::at(16 * R + r) + 4 * M) = x;
    if (row >= a.Sq) bits = 0;
    cw[r & 7] |= bits << (16 * (r >> 3));
  }
  transpose_16x16(cw);
#pragma unroll
  for (int t = 0; t < 16; t++)
    *reinterpret_cast<ACCT_LDS uint16_t*>(kb.col + KeepBlock::at(32 * M + 8 * (t >> 2) + 4 * g + (t & 3)) + 2 * R) = (uint16_t)(cw[t & 7] >> (16 * (t >> 3)));
  kb.store(a, rowbits, colbits);
}

hipError_t launch_drop_philox(const FaArgs& a, uint32_t* rowbits, uint32_t* colbits, hipStream_t st) {
  const long long nblk = (long long)a.B * a.N * a.Tr * ((a.Tc + 3) / 4);
  hipLaunchKernelGGL(fa_drop_philox_kernel, dim3((unsigned)nblk), dim3(256), 0, st, a, rowbits, colbits);
  return hipGetLastError();
}

hipError_t launch_drop_bits(const FaArgs& a, uint32_t* rowbits, uint32_t* colbits, hipStream_t st) {
  const long long nblk = (long long)a.B * a.N * a.Tr * ((a.Tc + 3) / 4);
  if (a.drop_es == 2) hipLaunchKernelGGL(fa_drop_bits_kernel<2>, dim3((unsigned)nblk), dim3(256), 0, st, a, rowbits, colbits);
  else hipLaunchKernelGGL(fa_drop_bits_kernel<1>, dim3((unsigned)nblk), dim3(256), 0, st, a, rowbits, colbits);
  return hipGetLastError();
}

hipError_t launch_mask_blocks(const FaArgs& a, uint8_t* flags, uint32_t* colbits, int MB, hipStream_t st) {
  const dim3 grid((unsigned)((long long)MB * a.Tr * a.Tc));
  uint8_t* tails = flags + (size_t)MB * a.Tr * a.Tc;    // (the key-tail table follows the classes)
  if (a.mask_es == 2) hipLaunchKernelGGL(fa_mask_prepass_kernel<2>, grid, dim3(256), 0, st, a, flags, tails, colbits);
  else hipLaunchKernelGGL(fa_mask_prepass_kernel<1>, grid, dim3(256), 0, st, a, flags, tails, colbits);
  return hipGetLastError();
}

}  // namespace acct
