// FP32 triangle attention forward (inference) on gfx950 MFMA.
//
//   out[b,o,q,h,:] = sum_k softmax_k(scale <q, k> + mask[b,o,k] + bias[bb,h,q,k]) v[k,:]
//
// in FP32: products of three-way bf16 splits on the bf16 matrix cores, within
// half a unit in the last place of the f32 products (split_f32.hpp), f32 sums
// and softmax; the contract of the reference's inference-only FP32 path
// (openfold3/core/kernels/turbopairformer/turbopairformer_attention_fp32.py:139-224):
// a row whose logits are all -inf produces zeros.
//
// Same schedule as the bf16 forward (csrc/attention.hip): one workgroup = 4
// waves x 32 queries of one plane, key tiles (64 keys for D <= 32, 32 above)
// double-buffered in LDS, the S^T = K Q^T accumulator of each 32-key block
// seeded with the prescaled, fragment-major bias, online softmax with a
// lazily raised running max, V^T operands through transposing reads.  K and V
// are split once per workgroup, when a tile is written to LDS (three bf16
// tiles each), Q once per wave, and P (finite, or NaN where a score is +inf or
// NaN) in registers on its way into the P V product.  A sequence that ends inside a tile reads zeros past N through the
// range of the buffer resources and masks those keys.
#include <type_traits>

#include "attn_tile.hpp"
#include "common.hpp"
#include "split_f32.hpp"
#include "tpf_status.hpp"

namespace tpf {

struct AttnGeomF {
  int B, O, H, N, D;
  int NP;                // N rounded up to 64: the pitch of the prescaled bias
  int64_t s_row;         // element stride between sequence rows of q/k/v
  int64_t s_head;        // element stride between heads of q/k/v
  int64_t bias_bstride;  // elements between bias batches (0 = shared)
  float scale;
};

// f32 bias -> f32 bias / scale in the fragment-major S^T layout (see the
// bf16 pre-pass in csrc/attention.hip).
__global__ __launch_bounds__(256) void attn_bias_prescale_f32_kernel(const float* __restrict__ bias,
                                                                     float* __restrict__ out,
                                                                     int64_t items, int N, int NP,
                                                                     float inv_scale) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (block, j, lane)
  if (i >= items) return;
  const int lane = (int)(i & 63), j = (int)((i >> 6) & 3);
  const int64_t blk = i >> 8;
  const int nkb = NP / 32;
  const int kb = (int)(blk % nkb);
  const int64_t hq = blk / nkb;
  const int qb = (int)(hq % nkb);
  const int64_t bh = hq / nkb;
  const int ql = lane & 31, hl = lane >> 5;
  const int qi = qb * 32 + ql, k0 = kb * 32 + 8 * j + 4 * hl;
  const float* src = bias + (bh * N + qi) * (int64_t)N + k0;
  f32x4 v;
  if (N == NP) {
    v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= inv_scale;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = qi < N && k0 + e < N ? src[e] * inv_scale : 0.f;
  }
  *reinterpret_cast<f32x4*>(out + i * 4) = v;
}

template <int DP, int KT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DP == 32 ? 3 : 2, 8))) void attn_fwd_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ mask, const float* __restrict__ bias_s, float* __restrict__ out,
    float* __restrict__ lse, AttnGeomF g) {
  constexpr int TE = KT * DP;         // elements of one tile
  constexpr int CH = DP / 4;          // 16-byte chunks per f32 row
  constexpr int PER = KT * CH / 256;  // K (and V) chunks per thread per tile
  constexpr int NB = KT / 32;         // 32-key blocks per tile
  static_assert(KT * CH % 256 == 0, "a tile's chunks split evenly over the threads");
  __shared__ __attribute__((aligned(16))) __bf16 KVs[2][2][3][TE];  // [buffer][K, V][h, m, l]

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int ql = lane & 31, hl = lane >> 5;
  const int N = g.N, NP = g.NP, D = g.D;
  const int qtiles = (N + 127) / 128;
  int64_t T;
  {
    const int64_t total = (int64_t)qtiles * g.H * g.B * g.O;
    const int64_t L = blockIdx.x, per = (total + 7) / 8;
    T = (L % 8) * per + L / 8;
    if (T >= total) return;
  }
  const int qt = (int)(T % qtiles);
  const int64_t rr = T / qtiles;
  const int plane = (int)(rr % ((int64_t)g.B * g.O));
  const int h = (int)(rr / ((int64_t)g.B * g.O));
  const int b = plane / g.O;
  const int q0 = qt * 128 + w * 32;
  const bool active = q0 < N;
  const int qi = q0 + ql;
  const bool qok = qi < N;

  const int64_t plane_off = (int64_t)plane * g.H * N * D + (int64_t)h * g.s_head;
  const int nblk = NP / 32, ntiles = (N + KT - 1) / KT;
  const float c2 = g.scale * kLog2e;
  const float inv_scale = 1.f / g.scale;
  const float thr = 8.f / c2;

  // Q rows (B operand of S^T = K Q^T), split; zeros past D and N.
  Split8 qs[DP / 16];
  {
    const float* qrow = q + plane_off + (int64_t)(qok ? qi : 0) * g.s_row;
#pragma unroll
    for (int s = 0; s < DP / 16; ++s) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int d0 = 16 * s + 8 * hl + 4 * u;
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
        if (qok && d0 < D) y = *reinterpret_cast<const f32x4*>(qrow + d0);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * u + e] = y[e];
      }
      bool ok;
      qs[s] = split8(x, &ok);
      if (!__all(ok)) qs[s] = split8<true>(x);
    }
  }
  // K / V chunk it of this thread: row (it * 256 + tid) / CH of the tile.  The
  // resource of a tile starts at its first row and ends with row N - 1.
  const int64_t row_bytes = g.s_row * 4;
  uint32_t vkv[PER];
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int idx = it * 256 + tid, c = idx % CH;
    vkv[it] = c * 4 < D ? (uint32_t)((idx / CH) * row_bytes + c * 16) : kBufOOB;
  }
  f32x4 kr[PER], vr[PER];
  auto load_kv = [&](int t) {
    // Tiles past the last one reload the last one (never consumed).
    const int64_t r0 = (int64_t)min(t, ntiles - 1) * KT;
    const int64_t left = (N - 1 - r0) * row_bytes + (int64_t)D * 4;
    const int bytes = (int)(left < 0x7FFFFFFF ? left : 0x7FFFFFFF);
    const __amdgpu_buffer_rsrc_t rk = raw_rsrc(k + plane_off + r0 * g.s_row, bytes);
    const __amdgpu_buffer_rsrc_t rv = raw_rsrc(v + plane_off + r0 * g.s_row, bytes);
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      kr[it] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, vkv[it], 0, 0));
      vr[it] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, vkv[it], 0, 0));
    }
  };
  auto store_split = [&](int buf, auto all) {  // whether the split served every element
    bool ok = true;
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int idx = it * 256 + tid;
      const int off = kv_off<DP>(idx / CH, 4 * (idx % CH));
      bool okk, okv;
      const Split4 ks = split4<decltype(all)::value>(kr[it], &okk);
      const Split4 vs = split4<decltype(all)::value>(vr[it], &okv);
      ok &= okk & okv;
      *reinterpret_cast<bf16x4*>(&KVs[buf][0][0][off]) = ks.h;
      *reinterpret_cast<bf16x4*>(&KVs[buf][0][1][off]) = ks.m;
      *reinterpret_cast<bf16x4*>(&KVs[buf][0][2][off]) = ks.l;
      *reinterpret_cast<bf16x4*>(&KVs[buf][1][0][off]) = vs.h;
      *reinterpret_cast<bf16x4*>(&KVs[buf][1][1][off]) = vs.m;
      *reinterpret_cast<bf16x4*>(&KVs[buf][1][2][off]) = vs.l;
    }
    return ok;
  };
  auto store_kv = [&](int buf) {
    if (!__all(store_split(buf, std::false_type{}))) store_split(buf, std::true_type{});
  };
  const __amdgpu_buffer_rsrc_t rs_b = raw_rsrc(
      bias_s + (int64_t)b * g.bias_bstride +
      ((int64_t)h * nblk + (active ? q0 / 32 : 0)) * (int64_t)nblk * 1024);
  auto load_bias = [&](int blk) {
    const uint32_t so = (uint32_t)min(blk, nblk - 1) * 4096;
    f32x16 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 x = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_b, (uint32_t)lane * 16 + j * 1024, so, 0));
#pragma unroll
      for (int i = 0; i < 4; ++i) r[4 * j + i] = x[i];
    }
    return r;
  };
  load_kv(0);
  f32x16 bset = load_bias(0);
  // Flags of the 64-key groups with any nonzero mask entry (keys past N
  // count); groups past the first 64 are taken as masked.
  const float* mrow = mask + (int64_t)plane * N;
  const __amdgpu_buffer_rsrc_t rs_m = raw_rsrc(mrow, N * 4);
  uint64_t mbits = ~0ull;
  if (NP <= 64 * 64) {
    mbits = 0ull;
    for (int t = 0; t < NP / 64; t += 4) {
      float mv[4];  // four groups' loads in flight per ballot round
#pragma unroll
      for (int u = 0; u < 4; ++u) mv[u] = buf_ldf(rs_m, (uint32_t)((t + u) * 64 + lane) * 4);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int key = (t + u) * 64 + lane;
        if (key >= N && key < NP) mv[u] = -INFINITY;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (__any(mv[u] != 0.f)) mbits |= 1ull << ((t + u) & 63);
    }
  }
  store_kv(0);

  f32x16 acc[DP / 32];
#pragma unroll
  for (int i = 0; i < DP / 32; ++i) acc[i] = zero16();
  float m = -INFINITY, l = 0.f, nm = 0.f;

  auto block = [&](int buf, int sb, int blk) {
    f32x16 s = bset;
#pragma unroll
    for (int ks = 0; ks < DP / 16; ++ks) {
      const int off = kv_off<DP>(sb * 32 + ql, 16 * ks + 8 * hl);
      const Split8 kf{*reinterpret_cast<const bf16x8*>(&KVs[buf][0][0][off]),
                      *reinterpret_cast<const bf16x8*>(&KVs[buf][0][1][off]),
                      *reinterpret_cast<const bf16x8*>(&KVs[buf][0][2][off])};
      s = mfma32_split(kf, qs[ks], s);
    }
    bset = load_bias(blk + 1);
    if ((mbits >> ((blk >> 1) & 63)) & 1ull) {
      f32x4 mv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        mv[j] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_m, (8 * j + 4 * hl) * 4, blk * 128, 0));
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s[4 * j + i] = blk * 32 + 8 * j + 4 * hl + i < N ? fmaf(mv[j][i], inv_scale, s[4 * j + i])
                                                           : -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = xor32_max(mx);
    if (__any(mx > m + thr)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = (m_new == -INFINITY) ? 1.f : fast_exp2((m - m_new) * c2);
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DP / 32; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
      m = m_new;
      nm = (m == -INFINITY) ? 0.f : -m * c2;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = fast_exp2(fmaf(s[8 * t + e], c2, nm));
        l += p[e];
      }
      const Split8 ps = split8(p);
      const int k0 = sb * 32 + 16 * t;
#pragma unroll
      for (int db = 0; db < DP / 32; ++db) {
        bf16x8 va[3];
#pragma unroll
        for (int u = 0; u < 3; ++u)
          va[u] = cat8(kv_tr_col4<DP>(KVs[buf][1][u], k0, k0 + 4, 32 * db),
                       kv_tr_col4<DP>(KVs[buf][1][u], k0 + 8, k0 + 12, 32 * db));
        acc[db] = mfma32_split(Split8{va[0], va[1], va[2]}, ps, acc[db]);
      }
    }
  };
  // Waves and lanes past N compute on zero Q rows and store nothing.
#pragma unroll 1
  for (int t = 0; t < ntiles; ++t) {
    __syncthreads();
    if constexpr (NB == 1) load_kv(t + 1);
    block(t & 1, 0, NB * t);
    if constexpr (NB == 2) {
      load_kv(t + 1);
      block(t & 1, 1, 2 * t + 1);
    }
    // Buffer (t + 1) % 2 was last read in tile t - 1, before the barrier above.
    store_kv((t + 1) & 1);
  }
  if (!qok) return;
  // (Both lanes l and l ^ 32 hold the same query, so they return together.)
  const float l_tot = xor32_sum(l);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  float* orow = out + (((int64_t)plane * N + qi) * g.H + h) * D;
#pragma unroll
  for (int db = 0; db < DP / 32; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d0 = db * 32 + 8 * j + 4 * hl;
      if (d0 < D) {
        f32x4 o4;
#pragma unroll
        for (int i = 0; i < 4; ++i) o4[i] = acc[db][4 * j + i] * inv;
        *reinterpret_cast<f32x4*>(orow + d0) = o4;
      }
    }
  if (hl == 0 && lse) {
    lse[((int64_t)plane * g.H + h) * N + qi] =
        l_tot > 0.f ? (m * c2 + log2f(l_tot)) * kLn2 : -INFINITY;
  }
}

}  // namespace tpf

using namespace tpf;

extern "C" {

int64_t tpf_attn_forward_f32_workspace_bytes(int64_t B, int64_t H, int64_t N,
                                             int64_t bias_batches) {
  (void)B;
  const int64_t NP = (N + 63) / 64 * 64;
  return bias_batches * H * NP * NP * 4;
}

int tpf_attn_forward_f32(const float* q, const float* k, const float* v, const float* mask,
                         const float* bias, float* out, float* lse, void* workspace,
                         int64_t workspace_bytes, int64_t B, int64_t O, int64_t H, int64_t N,
                         int64_t D, int layout, int64_t bias_batches, double scale,
                         void* stream) {
  const char* fn = "tpf_attn_forward_f32";
  if (layout & ~(TPF_QKV_SEQ_MAJOR | TPF_ANY_N))
    return set_error(TPF_ERR_ARG,
                     "%s: layout flags 0x%x: only TPF_QKV_SEQ_MAJOR and TPF_ANY_N are supported",
                     fn, layout);
  const bool seq_major = layout & TPF_QKV_SEQ_MAJOR;
  if (!q || !k || !v || !mask || !bias || !out || !workspace)
    return set_error(TPF_ERR_ARG, "%s: null pointer", fn);
  if (B < 1 || O < 1 || H < 1 || N < 1)
    return set_error(TPF_ERR_SHAPE, "%s: B, O, H and N must be positive", fn);
  if (N % 64 != 0 && !(layout & TPF_ANY_N))
    return set_error(TPF_ERR_SHAPE, "%s: N=%lld must be a multiple of 64 (pad on the host)", fn,
                     (long long)N);
  if (D < 4 || D > 64 || D % 4 != 0)
    return set_error(TPF_ERR_SHAPE, "%s: D=%lld must be a multiple of 4 in [4, 64]", fn,
                     (long long)D);
  if (bias_batches != 1 && bias_batches != B)
    return set_error(TPF_ERR_SHAPE, "%s: bias batch %lld must be 1 or B", fn,
                     (long long)bias_batches);
  if (workspace_bytes < tpf_attn_forward_f32_workspace_bytes(B, H, N, bias_batches))
    return set_error(TPF_ERR_ARG, "%s: workspace too small", fn);
  const int64_t total = ((N + 127) / 128) * H * B * O;
  if ((total + 7) / 8 * 8 > INT32_MAX || B * O > INT32_MAX)
    return set_error(TPF_ERR_SHAPE, "%s: too many query tiles", fn);
  AttnGeomF g;
  g.B = (int)B; g.O = (int)O; g.H = (int)H; g.N = (int)N; g.D = (int)D;
  g.s_row = seq_major ? H * D : D;
  g.s_head = seq_major ? D : N * D;
  const int64_t NP = (N + 63) / 64 * 64;
  g.NP = (int)NP;
  g.bias_bstride = (bias_batches == 1) ? 0 : H * NP * NP;
  g.scale = (float)scale;
  hipStream_t s = (hipStream_t)stream;
  float* bias_s = (float*)workspace;
  const int64_t items = bias_batches * H * NP * NP / 4;
  hipLaunchKernelGGL(attn_bias_prescale_f32_kernel, dim3((unsigned)((items + 255) / 256)),
                     dim3(256), 0, s, bias, bias_s, items, (int)N, (int)NP,
                     (float)(1.0 / scale));
  int rc = check_launch(fn);
  if (rc) return rc;
  dim3 grid((unsigned)((total + 7) / 8 * 8));
  if (D <= 32)
    hipLaunchKernelGGL((attn_fwd_f32_kernel<32, 64>), grid, dim3(256), 0, s, q, k, v, mask, bias_s, out,
                       lse, g);
  else
    hipLaunchKernelGGL((attn_fwd_f32_kernel<64, 32>), grid, dim3(256), 0, s, q, k, v, mask, bias_s, out,
                       lse, g);
  return check_launch(fn);
}

}  // extern "C"
