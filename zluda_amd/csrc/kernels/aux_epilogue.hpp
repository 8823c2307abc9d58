// Second, element-wise pass of the epilogues that keep or use the GELU input, for the problems whose GEMM kernel does not do it itself
// (aux_in_epilogue(); cuda_types/src/cublaslt.rs:4601-4660; the aux attributes :4182-4236):
//   GELU_AUX[_BIAS]  the GEMM kernel has written x = alpha * op(A) op(B) + beta * C (+ bias) into the aux matrix;
//                    this pass writes D = gelu(x) * d_scale
//   DGELU[_BGRAD]    the GEMM kernel has written y = alpha * op(A) op(B) + beta * C into D; this pass turns it into
//                    D = y * gelu'(aux) and, for _BGRAD, puts the sums of D's rows into the bias buffer
// aux is a matrix of D's type, shape and order.  Both passes see the value the first pass rounded to that type
// (a 16- or 32-bit float type; the planner admits no other here), so D can differ from a single-pass result by
// one more rounding of that type.
// Memory bound: both matrices once, in 16-byte pieces where base, pitch and batch stride allow (`wide`).
#pragma once
#include "bgrad_reduce.hpp"

namespace zluda_amd {

template <uint32_t TYPE>
__device__ __forceinline__ v4u32 piece_of_elems(const float *x) {
  v4u32 p;
#pragma unroll
  for (int d = 0; d < 4; d++)
    p[d] = TYPE == CUDA_R_32F ? f2bits(x[d]) : TYPE == CUDA_R_16BF ? pack_bf16x2(x[2 * d], x[2 * d + 1]) : pack_f16x2(x[2 * d], x[2 * d + 1]);
  return p;
}

struct AuxParams {
  void *D, *aux;
  int32_t NP, NQ, batch;         // P: D's unit-stride index
  int64_t d_sq, d_sb, aux_sq, aux_sb;
  const void *d_scale;
  int32_t wide;                  // every 16-byte piece of both matrices is aligned
  // DGELU_BGRAD, sums along Q (column-major D): as BgradParams
  int32_t per_block, sums;
  void *part, *out;
  uint32_t out_type;
  int64_t out_sb;
};

// `use(base of the piece's elements, values of D, values of aux)` -> what D becomes, on the V elements at (p0, q)
template <uint32_t TYPE, bool READ_D, class F>
__device__ __forceinline__ void aux_piece(const AuxParams &prm, int p0, int q, int bt, F &&use) {
  constexpr int V = elems16(TYPE), ESZ = 16 / V;
  const int64_t di = prm.d_sb * bt + (int64_t)q * prm.d_sq + p0, ai = prm.aux_sb * bt + (int64_t)q * prm.aux_sq + p0;
  float d[V], a[V];
  const bool whole = prm.wide && p0 + V <= prm.NP;
  if (whole) {
    const v4u32 ap = *(const v4u32 *)((const char *)prm.aux + ai * ESZ);
    v4u32 dp = v4u32{0, 0, 0, 0};
    if constexpr (READ_D) dp = *(const v4u32 *)((const char *)prm.D + di * ESZ);
#pragma unroll
    for (int e = 0; e < V; e++) { a[e] = elem_of_piece<TYPE>(ap, e); d[e] = elem_of_piece<TYPE>(dp, e); }
  } else {
#pragma unroll
    for (int e = 0; e < V; e++) {
      const bool in = p0 + e < prm.NP;
      a[e] = in ? load_elem(prm.aux, TYPE, ai + e) : 0.0f;
      d[e] = READ_D && in ? load_elem(prm.D, TYPE, di + e) : 0.0f;
    }
  }
  use(d, a);
  if (whole) {
    *(v4u32 *)((char *)prm.D + di * ESZ) = piece_of_elems<TYPE>(d);
  } else {
#pragma unroll
    for (int e = 0; e < V; e++)
      if (p0 + e < prm.NP) store_elem(prm.D, TYPE, di + e, d[e]);
  }
}

// grid (ceil(pieces / 256), 1, batch): one piece per thread (8192 x 4096 bf16: 81 us with one element per thread, 22 us now)
template <uint32_t TYPE>
__global__ __launch_bounds__(256) void aux_gelu_kernel(AuxParams prm) {
  constexpr int V = elems16(TYPE);
  const uint32_t ppr = (uint32_t)(prm.NP + V - 1) / V;
  const uint64_t x = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (x >= (uint64_t)ppr * prm.NQ) return;
  const int q = (int)(x / ppr), p0 = (int)(x % ppr) * V;
  const float sd = prm.d_scale ? *(const float *)prm.d_scale : 1.0f;
  aux_piece<TYPE, false>(prm, p0, q, blockIdx.z, [&](float (&d)[V], const float (&a)[V]) {
#pragma unroll
    for (int e = 0; e < V; e++) d[e] = gelu_tanh(a[e]) * sd;
  });
}

// Sums along Q, or none: 512 threads, LANES side by side along P; grid (ceil(NP / (LANES * V)), shares of Q, batch).
// (8192 x 4096 bf16 with row sums: 849 us one element at a time with a workgroup per 64 rows, 52 us now)
template <uint32_t TYPE, int LANES>
__global__ __launch_bounds__(512) void aux_dgelu_kernel(AuxParams prm) {
  constexpr int V = elems16(TYPE), PH = 512 / LANES;
  __shared__ float lds[512 * V];
  const int lane = threadIdx.x % LANES, phase = threadIdx.x / LANES, bt = blockIdx.z;
  const int p0 = (blockIdx.x * LANES + lane) * V;
  const int q1 = min(prm.NQ, ((int)blockIdx.y + 1) * prm.per_block);
  float s[V];
#pragma unroll
  for (int e = 0; e < V; e++) s[e] = 0.0f;
  if (p0 < prm.NP) {
#pragma unroll 2
    for (int q = (int)blockIdx.y * prm.per_block + phase; q < q1; q += PH)
      aux_piece<TYPE, true>(prm, p0, q, bt, [&](float (&d)[V], const float (&a)[V]) {
#pragma unroll
        for (int e = 0; e < V; e++) {
          d[e] *= dgelu_tanh(a[e]);
          s[e] += d[e];
        }
      });
  }
  if (!prm.sums) return;
  sum_phases<V>(s, lds, lane, phase, LANES, [&](int o, float total) {
    const int p = blockIdx.x * LANES * V + o;
    if (p >= prm.NP) return;
    if (gridDim.y > 1) ((float *)prm.part)[((int64_t)bt * gridDim.y + blockIdx.y) * prm.NP + p] = total;
    else store_elem(prm.out, prm.out_type, (int64_t)bt * prm.out_sb + p, total);
  });
}

// Sums along P (row-major D): one workgroup per Q index; grid (NQ, 1, batch)
template <uint32_t TYPE>
__global__ __launch_bounds__(256) void aux_dgelu_rows_kernel(AuxParams prm) {
  constexpr int V = elems16(TYPE);
  __shared__ float part[4];
  const int q = blockIdx.x, bt = blockIdx.z;
  float s = 0.0f;
  for (int p0 = threadIdx.x * V; p0 < prm.NP; p0 += 256 * V)
    aux_piece<TYPE, true>(prm, p0, q, bt, [&](float (&d)[V], const float (&a)[V]) {
#pragma unroll
      for (int e = 0; e < V; e++) {
        d[e] *= dgelu_tanh(a[e]);
        s += d[e];  // (elements past the end are zero)
      }
    });
  if (!prm.sums) return;
#pragma unroll
  for (int off = 32; off; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) store_elem(prm.out, prm.out_type, (int64_t)bt * prm.out_sb + q, (part[0] + part[1]) + (part[2] + part[3]));
}

} // namespace zluda_amd
