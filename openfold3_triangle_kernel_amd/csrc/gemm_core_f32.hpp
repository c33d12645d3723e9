// FP32 GEMM main loop on the bf16 matrix cores (split_f32.hpp: every operand
// element as three bf16 values, six products; 256 threads = 4 waves per
// workgroup), for the inference-only FP32 paths.
//
//   acc(m, n) = sum_{k in [kbeg, kend)} A(m, k) * B(n, k)     (all f32)
//
// Tile 128 (m) x 128 (n) x 32 (k); wave w owns the 64 x 64 sub-tile
// (wm, wn) = (w >> 1, w & 1) as 2 x 2 accumulators in the 32x32 MFMA layout
//   acc[i][j] register r <-> m = 64 wm + 32 i + 8 (r / 4) + 4 (lane / 32) + r % 4,
//                            n = 64 wn + 32 j + lane % 32.
// The tiles stay f32 in LDS and a wave splits its fragments after reading
// them: 5.5 VALU instructions per element, about as many cycles as the 24
// MFMAs of a 16-deep step of the 2 x 2 blocks, and the two waves of a SIMD
// overlap them.
//
// Operands are read from HBM straight into LDS (buffer_load ... lds, zeros
// outside the tensor), two k-stages in flight.  Either operand may be
//   KC (K-contiguous): X[row * ld + k] -- LDS tile [128 rows][32 k], the
//      16-byte chunk c of row r stored at slot c ^ (r & 7);
//   MN (MN-contiguous): X[k * ld + row] -- LDS tile [32 k][128 rows],
//      fragments are 4-byte reads of consecutive rows.
// A KC operand may take its rows through a map (RowMap): the TriMul input
// projection walks the positions of padded planes, in the transposed pair
// order for the incoming direction.
#pragma once

#include "common.hpp"
#include "split_f32.hpp"

namespace tpf {

constexpr int kFM = 128, kFN = 128, kFK = 32;
constexpr int kFTileBytes = kFM * kFK * 4;       // 16 KiB
constexpr int kFStageBytes = 2 * kFTileBytes;
constexpr int kFMainLdsBytes = 2 * kFStageBytes;  // 64 KiB

// Natural pair row of position m = (b*n + i)*np + k of planes of n rows of
// np >= n positions: (b, i, k), or (b, k, i) when transposed; -1 for the pad
// positions k >= n.
struct RowMap {
  int n = 0, np = 0, transposed = 0;  // n = 0: identity
  FastDiv div_np{}, div_ps{};         // division by np and n * np
  __device__ __forceinline__ int64_t row(uint32_t m) const {
    if (n == 0) return m;
    const uint32_t b = fdiv(m, div_ps), p = m - b * div_ps.d;
    const uint32_t i = fdiv(p, div_np), k = p - i * (uint32_t)np;
    if (k >= (uint32_t)n) return -1;
    return (int64_t)b * n * n + (transposed ? (int64_t)k * n + i : (int64_t)i * n + k);
  }
};

struct GemmOperandF32 {
  const float* p;  // element (0, 0) of this batch item
  int64_t ld;      // leading dimension in elements
  int rows;        // extent of the m (or n) dimension
  RowMap map = {};  // KC only
};

template <bool KC>
struct TileLoaderF32 {
  i32x4 rsrc;
  uint32_t row_off[4];  // KC: byte offset of each row start (kBufOOB if absent)
  int sub;              // KC: k offset of this lane; MN: k-row in instruction
  int col_ok;
  uint32_t col_off;
  int64_t ld;

  __device__ __forceinline__ void init(const GemmOperandF32& op, int r0) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    rsrc = buffer_rsrc(op.p);
    ld = op.ld;
    if (KC) {
      const int rin = lane >> 3;                  // 8 rows of 128 bytes per instruction
      sub = 4 * ((lane & 7) ^ (rin & 7));
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int row = r0 + 8 * (4 * w + t) + rin;
        uint32_t off = kBufOOB;
        const int64_t prow = row < op.rows ? op.map.row((uint32_t)row) : -1;
        if (prow >= 0) off = (uint32_t)(prow * op.ld * 4);
        row_off[t] = off;
      }
    } else {
      sub = lane >> 5;                            // 2 k-rows of 512 bytes per instruction
      const int col = r0 + 4 * (lane & 31);
      col_ok = col < op.rows;
      col_off = (uint32_t)col * 4;
    }
  }

  __device__ __forceinline__ void issue(int k0, int kend, char* tile) const {
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int j = 4 * w + t;
      uint32_t off;
      if (KC) {
        const int k = k0 + sub;
        off = (row_off[t] != kBufOOB && k < kend) ? row_off[t] + (uint32_t)k * 4 : kBufOOB;
      } else {
        const int k = k0 + 2 * j + sub;
        off = (col_ok && k < kend) ? (uint32_t)((int64_t)k * ld * 4) + col_off : kBufOOB;
      }
      buf2lds16(rsrc, off, tile + j * 1024);
    }
  }
};

// The eight k values 16 s + 8 (lane / 32) .. + 7 of row rbase + lane % 32, split.
template <bool KC, bool ALL>
__device__ __forceinline__ Split8 tile_frag_f32(const float* T, int rbase, int s) {
  const int lane = threadIdx.x & 63, hl = lane >> 5;
  const int r = rbase + (lane & 31);
  float v[8];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (KC) {
      const int slot = (4 * s + 2 * hl + u) ^ (r & 7);
      const f32x4 x = *reinterpret_cast<const f32x4*>(T + r * kFK + slot * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * u + e] = x[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * u + e] = T[(16 * s + 8 * hl + 4 * u + e) * kFM + r];
    }
  }
  return split8<ALL>(v);
}

// The tile's products with one kind of split (split_pair), the same on all
// threads: returns whether any sum of the tile is NaN.
template <bool A_KC, bool B_KC, bool ALL>
__device__ __forceinline__ bool gemm_tile_f32_pass(const GemmOperandF32& A,
                                                   const GemmOperandF32& B, int m0, int n0,
                                                   int kbeg, int kend, char* smem,
                                                   f32x16 (&acc)[2][2]) {
  __shared__ int nan_s[4];
  const int w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero16();
  TileLoaderF32<A_KC> la;
  TileLoaderF32<B_KC> lb;
  la.init(A, m0);
  lb.init(B, n0);
  const int nk = (kend - kbeg + kFK - 1) / kFK;
  if (nk <= 0) return false;
  la.issue(kbeg, kend, smem);
  lb.issue(kbeg, kend, smem + kFTileBytes);
  for (int kt = 0; kt < nk; ++kt) {
    char* cur = smem + (kt & 1) * kFStageBytes;
    wait_vmcnt<0>();
    lds_barrier();
    if (kt + 1 < nk) {
      char* nxt = smem + ((kt + 1) & 1) * kFStageBytes;
      la.issue(kbeg + (kt + 1) * kFK, kend, nxt);
      lb.issue(kbeg + (kt + 1) * kFK, kend, nxt + kFTileBytes);
    }
    const float* As = reinterpret_cast<const float*>(cur);
    const float* Bs = reinterpret_cast<const float*>(cur + kFTileBytes);
#pragma unroll
    for (int s = 0; s < kFK / 16; ++s) {
      Split8 af[2], bfr[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        af[t] = tile_frag_f32<A_KC, ALL>(As, 64 * wm + 32 * t, s);
        bfr[t] = tile_frag_f32<B_KC, ALL>(Bs, 64 * wn + 32 * t, s);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma32_split(af[i], bfr[j], acc[i][j]);
    }
  }
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) bad |= __builtin_isunordered(acc[i][0][r], acc[i][1][r]);
  const int any = __any(bad);
  if ((threadIdx.x & 63) == 0) nan_s[w] = any;
  lds_barrier();
  return __builtin_amdgcn_readfirstlane(nan_s[0] | nan_s[1] | nan_s[2] | nan_s[3]) != 0;
}

// Operands are taken to be finite floats below the largest bf16; where one is
// not, some sum is NaN, and the tile is formed again with the split that
// serves every float (no test of the operands in the main loop).
template <bool A_KC, bool B_KC>
__device__ __forceinline__ void gemm_tile_f32(const GemmOperandF32& A, const GemmOperandF32& B,
                                              int m0, int n0, int kbeg, int kend, char* smem,
                                              f32x16 (&acc)[2][2]) {
  if (gemm_tile_f32_pass<A_KC, B_KC, false>(A, B, m0, n0, kbeg, kend, smem, acc))
    gemm_tile_f32_pass<A_KC, B_KC, true>(A, B, m0, n0, kbeg, kend, smem, acc);
}

}  // namespace tpf
