// FlashAttention2 forward for ONE query row per head (gfx950): a new token against a key / value cache.
//
// Replaces the same builder as fa_fwd.hip (train/acctransformer/flash_attention/ops/flash_attention/flash_attention_fwd.py:308-474)
// where the query has one row, no mask tensor, no bias and no dropout.
//
// Bound by reading K and V once.  The tile kernel of fa_fwd.hip stages them through LDS in steps with a barrier and fills
// one row of 64 of its matrix tiles.  Here 16-byte chunks of the rows go from memory straight into registers, past the
// caches where nothing is read twice, 16 loads per wave in flight, and stay there: a row of K or V is spread over the CH lanes of a
// group, a wave holds 64 / CH rows per load, and every group keeps softmax statistics and sums of its own, in float32
// from the score to the sum (the probabilities are not rounded to the element type).  The groups meet at the end.
// Tile kernel / this one (us, bfloat16, caches read from memory): 256 heads, 3000 keys, D128 71.5 / 59.9 (6.6 TB/s); 384, 2000
// 85.8 / 62.8; 64, 1000, D64 13.0 / 8.6; 8, 8192, D128 18.0 / 13.6; 1, 131072 27.6 / 20.7; 64, 128, D64 5.1 / 5.2.  Error of O against 64
// bits 2.3e-3 / 1.7e-3 (bfloat16), 2.9e-4 / 2.1e-4 (float16): what is left is the rounding of O.
#include <type_traits>

#include "fa_common.hpp"
#include "fa_launch.hpp"

#ifndef ACCT_ELEM
#error "compiled once per element type: -DACCT_ELEM=f16 and -DACCT_ELEM=bf16"
#endif

namespace acct {

constexpr int kRowWaves = 8;

// sum over the pairs of two vectors of 8, products and sum in float32
ACCT_DEV float dot8(f16x8 a, f16x8 b) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) s = __builtin_amdgcn_fdot2(f16x2{a[2 * i], a[2 * i + 1]}, f16x2{b[2 * i], b[2 * i + 1]}, s, false);
  return s;
}
ACCT_DEV float dot8(bf16x8 a, bf16x8 b) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) s = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{a[2 * i], a[2 * i + 1]}, bf16x2{b[2 * i], b[2 * i + 1]}, s, false);
  return s;
}

// x of the lane at distance M, combined with the lane's own: every lane of the pair gets the same value
template <int M, typename F>
ACCT_DEV float with_lane(float x, F f) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8 || M == 16 || M == 32, "a power of two within the wave");
  if constexpr (M == 16) {
    const u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else if constexpr (M == 32) {
    const u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
  } else {
    // quad permutes for 1 and 2; the mirror image of 8 lanes serves 4, as the lanes below agree by then; a row turned by 8
    constexpr int ctrl = M == 1 ? 0xB1 : M == 2 ? 0x4E : M == 4 ? 0x141 : 0x128;
    return f(x, __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(x), ctrl, 0xf, 0xf, true)));
  }
}
// over the lanes of a group of CH (LO = 1) or over the groups of a wave (LO = CH, HI = 64)
template <int LO, int HI, typename F>
ACCT_DEV float over_lanes(float x, F f) {
  if constexpr (LO < HI) return over_lanes<2 * LO, HI>(with_lane<LO>(x, f), f);
  else return x;
}

// Whether workgroups of different heads or batches read the same lines of an operand: it is expanded over them, or heads lie
// beside each other in a row and do not end with a line of 128 bytes.  The loads then leave the lines in the caches.  Past the
// caches / through them (us, bfloat16): one K and V for all 32 heads, 16 batches, 8000 keys, D64 113 / 52 (tile kernel 85); 8
// batches, 3000, D128 37.7 / 22.8 (34.2); one for all batches, 4 x 64 heads, 8000, D128 86.7 / 59.9 (85.6); [B, S, N, D], 32 heads,
// 20000, D40 36.3 / 25.2 (47.1); 256, 4000, D80 80.1 / 77.1 (77.0).  Where nothing is shared, through them is slower: 256 heads, 3000,
// D128 61.0 / 67.6; 512, 8000, D64 164 / 177.
inline bool lines_are_shared(int extent, int64_t stride, int64_t row_stride, int hd) {
  return extent > 1 && stride < row_stride && (stride < hd || stride % 64 != 0);
}

// CH: 16-byte chunk slots per row (8, 16, 32 for head dims up to 64, 128, 256); KEEP: the loads leave their lines in the caches
template <typename T, int CH, bool KEEP>
__global__ void __launch_bounds__(64 * kRowWaves) fa_fwd_row_kernel(const FaArgs a, int key_end) {
  using E = Elem<T>;
  using V8 = typename E::V8;
  constexpr int R = 64 / CH, U = 4, NW = kRowWaves;          // rows per load, loads of K (and of V) per batch
  constexpr int STEP = NW * R * U;                           // rows per batch of the workgroup
  __shared__ float s_o[NW][CH * 8 + 2];
  const auto sum = [](float x, float y) { return x + y; };
  const auto larger = [](float x, float y) { return fmaxf(x, y); };
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane % CH, cpr = a.hd >> 3;
  const int parts = a.kv_split > 1 ? a.kv_split : 1;
  const uint32_t bh = blockIdx.x / (uint32_t)parts, part = blockIdx.x % (uint32_t)parts;
  const int64_t b = bh / (uint32_t)a.N, h = bh % (uint32_t)a.N;
  // this part's keys, in whole batches
  const int batches = (key_end + STEP - 1) / STEP;
  const int b_lo = (int)((uint32_t)batches * part / parts), b_hi = (int)((uint32_t)batches * (part + 1) / parts);   // (at most 2^23 batches, 256 parts)
  const int k_hi = min(b_hi * STEP, key_end);
  const int cc = min(c, cpr - 1);                            // (slots past the head dim repeat the last chunk, which does not count)
  const V8 q = *reinterpret_cast<const V8*>((const T*)a.q + b * a.q_sb + h * a.q_sh + cc * 8);
  const T* kp = (const T*)a.k + b * a.k_sb + h * a.k_sh;
  const T* vp = (const T*)a.v + b * a.v_sb + h * a.v_sh;
  const int lrow = lane / CH;                                // the lane's row within a load
  const uint32_t koff = (uint32_t)(lrow * a.k_ss + cc * 8) * 2, voff = (uint32_t)(lrow * a.v_ss + cc * 8) * 2;
  float m = -1e30f, l = 0.f, o[8];                           // (finite: all keys of a group may score -inf, and -inf - -inf is NaN)
#pragma unroll
  for (int e = 0; e < 8; e++) o[e] = 0.f;

  auto fetch = [](const void* p) {
    if constexpr (KEEP) return *reinterpret_cast<const V8*>(p);
    else return __builtin_nontemporal_load(reinterpret_cast<const V8*>(p));
  };
  auto load = [&](V8 (&kf)[U], V8 (&vf)[U], int batch) {
    const int row = batch * STEP + wave * (R * U);           // wave-uniform: a row's address is a scalar, the lane's part of it 32 bits
    if ((batch + 1) * STEP <= k_hi) {
#pragma unroll
      for (int u = 0; u < U; u++)
        kf[u] = fetch((const char*)(kp + (int64_t)(row + R * u) * a.k_ss) + koff);
#pragma unroll
      for (int u = 0; u < U; u++)
        vf[u] = fetch((const char*)(vp + (int64_t)(row + R * u) * a.v_ss) + voff);
    } else {                                                 // rows past the last key repeat it
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int64_t r = min(row + R * u + lrow, k_hi - 1);
        kf[u] = fetch(kp + r * a.k_ss + cc * 8);
        vf[u] = fetch(vp + r * a.v_ss + cc * 8);
      }
    }
  };
  auto work = [&](const V8 (&kf)[U], V8 (&vf)[U], int batch) {
    float s[U];
#pragma unroll
    for (int u = 0; u < U; u++) s[u] = over_lanes<1, CH>(c < cpr ? dot8(q, kf[u]) : 0.f, sum);
    if ((batch + 1) * STEP > k_hi) {                         // rows past the last key: no probability, and nothing of V
#pragma unroll
      for (int u = 0; u < U; u++)
        if (batch * STEP + wave * (R * U) + R * u + lrow >= k_hi) {
          s[u] = -INFINITY;
#pragma unroll
          for (int e = 0; e < 8; e++) vf[u][e] = 0;
        }
    }
    float mx = m;
#pragma unroll
    for (int u = 0; u < U; u++) mx = fmaxf(mx, s[u]);
    const float alpha = fast_exp2((m - mx) * a.scale_log2e), mc = mx * a.scale_log2e;
    m = mx;
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] *= alpha;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float p = fast_exp2(__builtin_fmaf(s[u], a.scale_log2e, -mc));
      l += p;
#pragma unroll
      for (int e = 0; e < 8; e++) o[e] = __builtin_fmaf(p, (float)vf[u][e], o[e]);
    }
  };
  if (b_lo < b_hi) {
    V8 k0[U], v0[U], k1[U], v1[U];
    load(k0, v0, b_lo);
    for (int batch = b_lo; batch < b_hi; batch += 2) {
      if (batch + 1 < b_hi) load(k1, v1, batch + 1);
      work(k0, v0, batch);
      if (batch + 1 < b_hi) {
        if (batch + 2 < b_hi) load(k0, v0, batch + 2);
        work(k1, v1, batch + 1);
      }
    }
  }
  // the groups of the wave, then the waves
  {
    const float mx = over_lanes<CH, 64>(m, larger), w = fast_exp2((m - mx) * a.scale_log2e);
    m = mx;
    l = over_lanes<CH, 64>(l * w, sum);
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = over_lanes<CH, 64>(o[e] * w, sum);
  }
  if (lane < CH) {
#pragma unroll
    for (int e = 0; e < 8; e++) s_o[wave][8 * c + e] = o[e];
    if (lane == 0) { s_o[wave][CH * 8] = m; s_o[wave][CH * 8 + 1] = l; }
  }
  __syncthreads();
  if (tid >= a.hd) return;
  float mm = s_o[0][CH * 8];
#pragma unroll
  for (int i = 1; i < NW; i++) mm = fmaxf(mm, s_o[i][CH * 8]);
  float lt = 0.f, ot = 0.f;
#pragma unroll
  for (int i = 0; i < NW; i++) {
    const float w = fast_exp2((s_o[i][CH * 8] - mm) * a.scale_log2e);
    lt = __builtin_fmaf(s_o[i][CH * 8 + 1], w, lt);
    ot = __builtin_fmaf(s_o[i][tid], w, ot);
  }
  if (parts > 1) {                                           // sums [part][head][hd], then (m, l) [part][head]
    const int64_t heads = (int64_t)a.B * a.N, at = part * heads + bh;
    a.fwd_part[at * a.hd + tid] = ot;
    if (tid == 0) *reinterpret_cast<f32x2*>(a.fwd_part + parts * heads * a.hd + 2 * at) = f32x2{mm, lt};
    return;
  }
  ((T*)a.o)[b * a.o_sb + h * a.o_sh + tid] = (T)(ot * (lt > 0.f ? 1.0f / lt : 0.f));     // (a NaN stays one)
  if (tid == 0) a.lse[bh] = lt > 0.f ? mm * a.scale + __logf(lt) : -INFINITY;
}

// The parts of a head added up: one workgroup per head, thread c + cols * g takes column c and every (512 / cols)-th part.
template <typename T>
__global__ void __launch_bounds__(512) fa_fwd_row_combine_kernel(const FaArgs a, int cols) {
  __shared__ float s_m[512], s_l[512], s_o[512];
  const int bh = blockIdx.x, tid = threadIdx.x, col = tid % cols, grp = tid / cols, groups = 512 / cols, parts = a.kv_split;
  const int64_t b = bh / a.N, h = bh % a.N, heads = (int64_t)a.B * a.N;
  const f32x2* stat = reinterpret_cast<const f32x2*>(a.fwd_part + parts * heads * a.hd);
  const int cc = min(col, a.hd - 1);
  float m = -1e30f, l = 0.f, o = 0.f;
  constexpr int U = 8;
  for (int s0 = grp; s0 < parts; s0 += groups * U) {
    float v[U];
    f32x2 ml[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t at = min(s0 + u * groups, parts - 1) * heads + bh;       // (a repeated part is left out below)
      v[u] = a.fwd_part[at * a.hd + cc];
      ml[u] = stat[at];
    }
    float mb = m;
#pragma unroll
    for (int u = 0; u < U; u++) mb = fmaxf(mb, ml[u][0]);
    const float al = fast_exp2((m - mb) * a.scale_log2e);
    m = mb;
    l *= al;
    o *= al;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = s0 + u * groups < parts;
      const float w = in ? fast_exp2((ml[u][0] - m) * a.scale_log2e) : 0.f;
      l = __builtin_fmaf(ml[u][1], w, l);
      o = __builtin_fmaf(in ? v[u] : 0.f, w, o);
    }
  }
  s_m[tid] = m; s_l[tid] = l; s_o[tid] = o;
  __syncthreads();
  if (tid >= a.hd) return;
  for (int g = 1; g < groups; g++) m = fmaxf(m, s_m[g * cols + tid]);
  l = 0.f;
  o = 0.f;
  for (int g = 0; g < groups; g++) {
    const float w = fast_exp2((s_m[g * cols + tid] - m) * a.scale_log2e);
    l = __builtin_fmaf(s_l[g * cols + tid], w, l);
    o = __builtin_fmaf(s_o[g * cols + tid], w, o);
  }
  ((T*)a.o)[b * a.o_sb + h * a.o_sh + tid] = (T)(o * (l > 0.f ? 1.0f / l : 0.f));
  if (tid == 0) a.lse[bh] = l > 0.f ? m * a.scale + __logf(l) : -INFINITY;
}

template <typename T>
hipError_t launch_fwd_row_elem(const FaArgs& a, int key_end, hipStream_t st) {
  const int ch = a.hd <= 64 ? 8 : a.hd <= 128 ? 16 : 32;
  const unsigned heads = (unsigned)(a.B * a.N);
  const bool keep = lines_are_shared(a.N, a.k_sh, a.k_ss, a.hd) || lines_are_shared(a.B, a.k_sb, a.k_ss, a.hd) ||
                    lines_are_shared(a.N, a.v_sh, a.v_ss, a.hd) || lines_are_shared(a.B, a.v_sb, a.v_ss, a.hd);
  auto pick = [&](auto k) {
    constexpr bool KEEP = decltype(k)::value;
    return ch == 8 ? fa_fwd_row_kernel<T, 8, KEEP> : ch == 16 ? fa_fwd_row_kernel<T, 16, KEEP> : fa_fwd_row_kernel<T, 32, KEEP>;
  };
  auto kern = keep ? pick(std::true_type{}) : pick(std::false_type{});
  hipLaunchKernelGGL(kern, dim3(heads * (a.kv_split > 1 ? a.kv_split : 1)), dim3(64 * kRowWaves), 0, st, a, key_end);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && a.kv_split > 1) {
    hipLaunchKernelGGL(fa_fwd_row_combine_kernel<T>, dim3(heads), dim3(512), 0, st, a, a.hd <= 64 ? 64 : a.hd <= 128 ? 128 : 256);
    e = hipGetLastError();
  }
  return e;
}
template hipError_t launch_fwd_row_elem<ACCT_ELEM>(const FaArgs& a, int key_end, hipStream_t st);

}  // namespace acct
