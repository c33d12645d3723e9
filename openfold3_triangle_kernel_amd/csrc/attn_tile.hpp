// K / V tiles of the attention forwards in LDS: rows of DP bf16, 16-byte
// chunks swizzled by the row.
#pragma once

#include "common.hpp"

namespace tpf {

// Swizzle of the 16-byte chunks of K / V tile rows: a 16-byte row read by 8
// consecutive rows (8 lanes = 128 bytes) and an 8-byte transposing read of 4
// consecutive rows x 2 chunks (16 lanes = 128 bytes) each cover all 32
// banks once.  DP = 32 (64-byte rows): rows 0..7 -> 0, 0, 2, 2, 1, 1, 3, 3;
// DP = 64 (128-byte rows): 0, 2, 4, 6, 1, 3, 5, 7.
template <int DP>
__device__ __forceinline__ int kv_swz(int r) {
  return (DP == 32) ? ((((r >> 1) & 1) << 1) | ((r >> 2) & 1)) : (((r & 3) << 1) | ((r >> 2) & 1));
}
template <int DP>
__device__ __forceinline__ int kv_off(int r, int col) {  // element offset of (row, col)
  return r * DP + (((col >> 3) ^ kv_swz<DP>(r)) << 3) + (col & 7);
}

// tr_col4 (common.hpp) on a swizzled K / V tile: lane l receives
// { M[r0 + e][c0 + l % 32] : e = 0..3 }, r0 = rbase_lo (l < 32) or rbase_hi.
template <int DP>
__device__ __forceinline__ bf16x4 kv_tr_col4(const __bf16* M, int rbase_lo, int rbase_hi, int c0) {
  const int l = threadIdx.x & 63, gq = l >> 4, ip = l & 15;
  const int r = ((gq >> 1) ? rbase_hi : rbase_lo) + (ip >> 2);
  const __bf16* p = M + kv_off<DP>(r, c0 + 16 * (gq & 1) + 4 * (ip & 3));
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}

}  // namespace tpf
