// The second kernel of a split-K matmul (see MfmaParams::splits in gemm_mfma.hpp).
#pragma once
#include "gemm_mfma.hpp"

namespace zluda_amd {

// Sums the partial tiles and applies the full epilogue (any D type,
// C read, vectors).  One thread per 4 consecutive elements along P; grid (ceil(NP / 1024), NQ, batch).
struct SplitKReduceParams {
  GemmArgs g;
  int32_t swapped, splits, acc_is_int;
  int32_t ws_np, ws_nq;  // padded extents of one partial matrix
  const int32_t *ws;
};
// Bound by latency, not by bytes (a partial tile or two per CU, a few us): what can be asked for at once is.
// SPLITS, the number of partial tiles, is a template argument (0: any number, one after the other), so that all of a thread's partial sums are on their
// way together with the vectors of the epilogue; the arguments, which lie in host memory, are fetched in one go (fetch_args() says
// why).  The sums run in the order of the
// shares.  (us of the whole call, before one load after the other: f32 468 x 310 x 938 in seven shares 13.9 -> 12.9, bf16
// 594 x 448 x 1615 in six 15.1 -> 12.8, 960 x 124 x 31971 in eight 49.2 -> 45.7.)
template <int SPLITS>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(SplitKReduceParams prm) {
#if defined(__HIP_DEVICE_COMPILE__)
  {
    constexpr int LINES = (sizeof(SplitKReduceParams) + 63) / 64;
    static_assert(LINES == 6, "one operand per line below");
    const uint32_t *w = (const uint32_t *)&prm;
    asm volatile("" ::"s"(w[0]), "s"(w[16]), "s"(w[32]), "s"(w[48]), "s"(w[64]), "s"(w[80]));
  }
#endif
  const GemmArgs &g = prm.g;
  const int NP = prm.swapped ? g.N : g.M;
  const int p = (blockIdx.x * 256 + threadIdx.x) * 4, q = blockIdx.y, bt = blockIdx.z;
  if (p >= NP) return;
  const int64_t plane = (int64_t)prm.ws_np * prm.ws_nq, step = g.batch * plane;
  const int32_t *src = prm.ws + (int64_t)bt * plane + (int64_t)q * prm.ws_np + p;
  v4i si;
  float sf[4];
  if constexpr (SPLITS > 0) {
    v4i t[SPLITS];
#pragma unroll
    for (int z = 0; z < SPLITS; z++) t[z] = *(const v4i *)(src + z * step);
    si = t[0];
#pragma unroll
    for (int e = 0; e < 4; e++) sf[e] = bits2f((uint32_t)si[e]);
#pragma unroll
    for (int z = 1; z < SPLITS; z++) {
      si += t[z];
#pragma unroll
      for (int e = 0; e < 4; e++) sf[e] += bits2f((uint32_t)t[z][e]);
    }
  } else {
    si = *(const v4i *)src;
#pragma unroll
    for (int e = 0; e < 4; e++) sf[e] = bits2f((uint32_t)si[e]);
    for (int z = 1; z < prm.splits; z++) {
      const v4i t = *(const v4i *)(src + z * step);
      si += t;
#pragma unroll
      for (int e = 0; e < 4; e++) sf[e] += bits2f((uint32_t)t[e]);
    }
  }
  Epilogue ep(g, bt);
  // (uniform) a float D without a C read, in one store where its four elements exist and are aligned
  if (!g.int_scale && g.beta_mode == SCALAR_VALUE && g.beta_val.f == 0.0f &&
      (g.d_type == CUDA_R_32F || g.d_type == CUDA_R_16F || g.d_type == CUDA_R_16BF)) {
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int pi = min(p + e, NP - 1), i = prm.swapped ? q : pi, j = prm.swapped ? pi : q;
      x[e] = ep.finish(ep.row_scale(i) * ep.col_scale(j) * (prm.acc_is_int ? (float)si[e] : sf[e]) + ep.bias_at(i));
    }
    const int64_t at = g.d_sb * bt + (int64_t)q * (prm.swapped ? g.d_si : g.d_sj) + p;
    if (g.d_type == CUDA_R_32F) {
      float *d = (float *)g.D + at;
      if (p + 3 < NP && (((uintptr_t)d) & 15) == 0) *(float4 *)d = make_float4(x[0], x[1], x[2], x[3]);
      else
#pragma unroll
        for (int e = 0; e < 4; e++) if (p + e < NP) d[e] = x[e];
    } else {
      uint16_t *d = (uint16_t *)g.D + at;
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; e++) h[e] = g.d_type == CUDA_R_16BF ? enc_bf16(x[e]) : enc_f16(x[e]);
      if (p + 3 < NP && (((uintptr_t)d) & 7) == 0) *(uint2 *)d = make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
      else
#pragma unroll
        for (int e = 0; e < 4; e++) if (p + e < NP) d[e] = h[e];
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    if (p + e >= NP) break;
    const int i = prm.swapped ? q : p + e, j = prm.swapped ? p + e : q;
    if (g.int_scale) ep.store_int(i, j, si[e]);
    else ep.store_f(i, j, prm.acc_is_int ? (float)si[e] : sf[e]);
  }
}

} // namespace zluda_amd
