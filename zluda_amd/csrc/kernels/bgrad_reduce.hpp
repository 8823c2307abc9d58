// Sums of matrix rows in two shapes, used by the bias-gradient epilogues as a small kernel behind the matmul:
//   CUBLASLT_EPILOGUE_BGRADA / BGRADB  the sums over the GEMM's K dimension of each row of op(A) (M values) or each column
//     of op(B) (N values); D is computed by the matmul kernel as with the DEFAULT epilogue
//   CUBLASLT_EPILOGUE_DGELU_BGRAD      the sums of D's rows, taken while D is turned into its gradient (aux_epilogue.hpp)
// Memory bound: one read of the matrix in 16-byte pieces.
#pragma once
#include "numeric.hpp"

namespace zluda_amd {

typedef uint32_t v4u32 __attribute__((ext_vector_type(4)));

// elements of TYPE in a 16-byte piece
constexpr int elems16(uint32_t type) { return type == CUDA_R_32F ? 4 : (type == CUDA_R_16F || type == CUDA_R_16BF) ? 8 : 16; }

template <uint32_t TYPE>
__device__ __forceinline__ float elem_of_piece(v4u32 p, int e) {
  if constexpr (TYPE == CUDA_R_32F) return bits2f(p[e]);
  else if constexpr (TYPE == CUDA_R_16BF) return (e & 1) ? bits2f(p[e >> 1] & 0xffff0000u) : bits2f(p[e >> 1] << 16);
  else if constexpr (TYPE == CUDA_R_16F) return dec_f16((uint16_t)(p[e >> 1] >> (16 * (e & 1))));
  else {
    const uint8_t b = (uint8_t)(p[e >> 2] >> (8 * (e & 3)));
    return TYPE == CUDA_R_8I ? (float)(int8_t)b : TYPE == CUDA_R_8F_E4M3 ? dec_e4m3(b) : dec_e5m2(b);
  }
}

struct BgradParams {
  const void *src;         // A or B
  int32_t rows, K, batch;  // `rows` sums of K elements per batch
  int64_t s_row, s_k, s_b; // element strides: row index, K, batch
  void *out;
  uint32_t out_type;
  int64_t out_sb;
  int32_t wide;            // 16-byte pieces: base, pitch and batch stride are multiples of 16 bytes
  // bgrad_cols_kernel: gridDim.y workgroups share a row's K, `per_block` each; with more than one of them the sums of each
  // go to part[batch][gridDim.y][rows] (fp32, int32 for int8 operands) and bgrad_finish_kernel adds them up
  int32_t per_block;
  void *part;
};

// K has the smaller stride: one workgroup per row, lanes run along K; grid (rows, 1, batch)
template <uint32_t TYPE>
__global__ __launch_bounds__(256) void bgrad_rows_kernel(BgradParams prm) {
  constexpr bool INTS = TYPE == CUDA_R_8I;  // summed exactly in int32, converted once
  constexpr int V = elems16(TYPE), ESZ = 16 / V;
  __shared__ float part_f[4];
  __shared__ int32_t part_i[4];
  const int r = blockIdx.x, bt = blockIdx.z;
  const int64_t base = (int64_t)bt * prm.s_b + (int64_t)r * prm.s_row;
  float s = 0.0f;
  int32_t si = 0;
  int k = threadIdx.x;
  if (prm.wide && prm.s_k == 1) {
    const int pieces = prm.K / V;
    for (int p = threadIdx.x; p < pieces; p += 256) {
      const v4u32 x = *(const v4u32 *)((const char *)prm.src + (base + (int64_t)p * V) * ESZ);
#pragma unroll
      for (int e = 0; e < V; e++) {
        if (INTS) si += (int8_t)(x[e >> 2] >> (8 * (e & 3)));
        else s += elem_of_piece<TYPE>(x, e);
      }
    }
    k += pieces * V;
  }
  for (; k < prm.K; k += 256) {
    if (INTS) si += ((const int8_t *)prm.src)[base + (int64_t)k * prm.s_k];
    else s += load_elem(prm.src, TYPE, base + (int64_t)k * prm.s_k);
  }
#pragma unroll
  for (int off = 32; off; off >>= 1) {
    si += __shfl_xor(si, off, 64);
    s += __shfl_xor(s, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    part_f[threadIdx.x >> 6] = s;
    part_i[threadIdx.x >> 6] = si;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const float total = INTS ? (float)(part_i[0] + part_i[1] + part_i[2] + part_i[3]) : (part_f[0] + part_f[1]) + (part_f[2] + part_f[3]);
    store_elem(prm.out, prm.out_type, (int64_t)bt * prm.out_sb + r, total);
  }
}

// Adds up what the 512 threads of a workgroup hold -- V consecutive sums each, `lanes` threads side by side, 512 / lanes of
// them behind each other (phases) -- and hands the totals of `lanes` * V consecutive rows to `put`.
template <int V, class T, class F>
__device__ __forceinline__ void sum_phases(T (&s)[V], T *lds, int lane, int phase, int lanes, F &&put) {
#pragma unroll
  for (int e = 0; e < V; e++) lds[phase * lanes * V + e * lanes + lane] = s[e];  // (lane-contiguous: no bank conflicts)
  __syncthreads();
  for (int o = threadIdx.x; o < lanes * V; o += 512) {
    T total = 0;
    for (int ph = 0; ph < 512 / lanes; ph++) total += lds[ph * lanes * V + o];
    put((o % lanes) * V + o / lanes, total);
  }
}

// The row index has the smaller stride: every step of the K walk reads consecutive rows; grid (ceil(rows / (LANES * V)), K shares, batch).
// One thread per row with a serial walk along K took 1442 us for 2048 rows of 4096 bf16 elements; 512 threads of 16-byte
// pieces per group of rows, four pieces in flight per thread, and K shared out over workgroups while there is scratch for
// their sums: 5.6 us and 4.9 for the second kernel.
template <uint32_t TYPE, int LANES>
__global__ __launch_bounds__(512) void bgrad_cols_kernel(BgradParams prm) {
  constexpr bool INTS = TYPE == CUDA_R_8I;
  constexpr int V = elems16(TYPE), ESZ = 16 / V, PH = 512 / LANES;
  using sum_t = typename std::conditional<INTS, int32_t, float>::type;
  __shared__ sum_t lds[512 * V];
  const int lane = threadIdx.x % LANES, phase = threadIdx.x / LANES, bt = blockIdx.z;
  const int r0 = (blockIdx.x * LANES + lane) * V;
  const int k0 = blockIdx.y * prm.per_block, k1 = min(prm.K, k0 + prm.per_block);
  const int64_t base = (int64_t)bt * prm.s_b + (int64_t)r0 * prm.s_row;
  sum_t s[V];
#pragma unroll
  for (int e = 0; e < V; e++) s[e] = 0;
  if (prm.wide && prm.s_row == 1 && r0 + V <= prm.rows) {
    auto add = [&](v4u32 x) {
#pragma unroll
      for (int e = 0; e < V; e++) {
        if constexpr (INTS) s[e] += (int8_t)(x[e >> 2] >> (8 * (e & 3)));
        else s[e] += elem_of_piece<TYPE>(x, e);
      }
    };
    const char *src = (const char *)prm.src + base * ESZ;
    int k = k0 + phase;
    for (; k + 3 * PH < k1; k += 4 * PH) {
      v4u32 x[4];
#pragma unroll
      for (int u = 0; u < 4; u++) x[u] = *(const v4u32 *)(src + (int64_t)(k + u * PH) * prm.s_k * ESZ);
#pragma unroll
      for (int u = 0; u < 4; u++) add(x[u]);
    }
    for (; k < k1; k += PH) add(*(const v4u32 *)(src + (int64_t)k * prm.s_k * ESZ));
  } else {
    for (int k = k0 + phase; k < k1; k += PH)
#pragma unroll
      for (int e = 0; e < V; e++)
        if (r0 + e < prm.rows) {
          const int64_t idx = base + e * prm.s_row + (int64_t)k * prm.s_k;
          if constexpr (INTS) s[e] += ((const int8_t *)prm.src)[idx];
          else s[e] += load_elem(prm.src, TYPE, idx);
        }
  }
  sum_phases<V>(s, lds, lane, phase, LANES, [&](int o, sum_t total) {
    const int r = blockIdx.x * LANES * V + o;
    if (r >= prm.rows) return;
    if (gridDim.y > 1) ((sum_t *)prm.part)[((int64_t)bt * gridDim.y + blockIdx.y) * prm.rows + r] = total;
    else store_elem(prm.out, prm.out_type, (int64_t)bt * prm.out_sb + r, (float)total);
  });
}

// The sums of the `shares` workgroups (or waves) of a row, added in their order; grid (ceil(rows / ROWS), 1, batch), PHASES threads a row.
struct BgradFinishParams {
  const void *part;  // [batch][shares][rows]
  int32_t shares, rows, ints;
  void *out;
  uint32_t out_type;
  int64_t out_sb;
};
template <int ROWS, int PHASES>
__global__ __launch_bounds__(ROWS *PHASES) void bgrad_finish_kernel(BgradFinishParams prm) {
  __shared__ float pf[ROWS * PHASES];
  __shared__ int32_t pi[ROWS * PHASES];
  const int t = threadIdx.x % ROWS, r = blockIdx.x * ROWS + t, phase = threadIdx.x / ROWS, bt = blockIdx.z;
  float s = 0.0f;
  int32_t si = 0;
  if (r < prm.rows) {
    const int64_t base = (int64_t)bt * prm.shares * prm.rows + r;
    const int per = (prm.shares + PHASES - 1) / PHASES, y1 = min(prm.shares, (phase + 1) * per);
#pragma unroll 8
    for (int y = phase * per; y < y1; y++) {
      const uint32_t raw = ((const uint32_t *)prm.part)[base + (int64_t)y * prm.rows];
      si += (int32_t)raw;
      s += bits2f(raw);
    }
  }
  pf[threadIdx.x] = s;
  pi[threadIdx.x] = si;
  __syncthreads();
  if (phase == 0 && r < prm.rows) {
    float qf[4];
    int32_t qi[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {  // a quarter of the phases each
      qf[q] = pf[q * (PHASES / 4) * ROWS + t];
      qi[q] = pi[q * (PHASES / 4) * ROWS + t];
#pragma unroll
      for (int ph = 1; ph < PHASES / 4; ph++) {
        qf[q] += pf[(q * (PHASES / 4) + ph) * ROWS + t];
        qi[q] += pi[(q * (PHASES / 4) + ph) * ROWS + t];
      }
    }
    const float total = prm.ints ? (float)(qi[0] + qi[1] + qi[2] + qi[3]) : (qf[0] + qf[1]) + (qf[2] + qf[3]);
    store_elem(prm.out, prm.out_type, (int64_t)bt * prm.out_sb + r, total);
  }
}

} // namespace zluda_amd
