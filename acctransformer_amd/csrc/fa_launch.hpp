// Host-side launchers of the gfx950 attention kernels (one per translation unit).
#pragma once
#include "fa_common.hpp"

#include <mutex>
#include <set>
#include <utility>

namespace acct {

// Raises a kernel's dynamic LDS limit once per (kernel, device) instead of on every launch.
inline hipError_t allow_dynamic_lds(const void* kern, size_t bytes) {
  static std::mutex mu;
  static std::set<std::pair<const void*, int>> done;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  if (done.count({kern, dev})) return hipSuccess;
  e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) done.insert({kern, dev});
  return e;
}

// forward: kg = key groups of the workgroup (FwdPlan, fa_index_math.hpp); the bias / dropout variants are picked from
// a.alibi / a.droprow, the key-range split from a.kv_split / a.fwd_part
template <typename T> hipError_t launch_fwd_elem(const FaArgs& a, int D, int kg, hipStream_t st);

// forward with one query row per head, the keys 0 .. key_end - 1 and no side inputs (fa_fwd_row.hip); a.kv_split / a.fwd_part:
// parts of the key range (RowPlan, fa_index_math.hpp)
template <typename T> hipError_t launch_fwd_row_elem(const FaArgs& a, int key_end, hipStream_t st);

// backward: delta pre-pass, dK/dV kernel (kv-tile owner) and dQ kernel (q-tile owner)
enum : int { kStageDq = 1, kStageDkDv = 2 };
template <typename T> hipError_t launch_bwd_elem(const FaArgs& a, int D, int stages, hipStream_t st);

// the dQ kernel with 64 query rows per wave (fa_bwd_dq64.hip): head dim 128, no side inputs, aligned lengths
bool dq64_applicable(const FaArgs& a);
hipError_t launch_bwd_dq64(FaArgs a, int dtype, hipStream_t st);

// false when the kernel translation units were compiled with a reduced variant set (ACCT_DEV_BUILD: head dim 128
// without side inputs)
#ifdef ACCT_DEV_BUILD
constexpr bool launch_variants_complete() { return false; }
#else
constexpr bool launch_variants_complete() { return true; }
#endif

// classify the 128x128 blocks of a dense mask into clean / apply / skip / causal diagonal, fill the key-tail table behind
// the classes and, with `colbits` non-null, pack the 'apply' blocks into per-key-column bitmaps [MB, Tr, Sk, 4 x u32]
hipError_t launch_mask_blocks(const FaArgs& a, uint8_t* flags, uint32_t* colbits, int MB, hipStream_t st);
// pack the dropout mask into keep bits by query row [B*N, Sq, droprow_w] and / or by key column [B*N, Tr, Sk, 4]
hipError_t launch_drop_bits(const FaArgs& a, uint32_t* rowbits, uint32_t* colbits, hipStream_t st);
// the same two bitmaps generated from (a.philox_k0, a.philox_k1, a.philox_offset, a.philox_thr) instead of read from a mask
hipError_t launch_drop_philox(const FaArgs& a, uint32_t* rowbits, uint32_t* colbits, hipStream_t st);
// the compact tile packed by key column: out[key][4]
hipError_t launch_mask_tilebits(const FaArgs& a, uint32_t* out, hipStream_t st);

}  // namespace acct
