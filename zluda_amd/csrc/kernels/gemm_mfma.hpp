// Shared pieces of the MFMA GEMM kernels for K-contiguous operands on gfx950 (CDNA4): vector types,
// LDS swizzle, direct global -> LDS copies, and the fused epilogues.  The K loop is in
// gemm_mfma_pipe.hpp.
//
//   KIND_I8   : int8 x int8 -> int32         v_mfma_i32_32x32x32_i8
//   KIND_F8   : e4m3/e5m2 -> fp32            v_mfma_f32_32x32x64_f8f6f4 (formats FP/FQ)
//   KIND_MXF4 : e2m1 + UE8M0 per 32 -> fp32  v_mfma_scale_f32_32x32x64_f8f6f4 (cbsz=blgp=4)
//   KIND_F16  : f16 x f16 -> fp32            v_mfma_f32_32x32x16_f16
//   KIND_BF16 : bf16 x bf16 -> fp32          v_mfma_f32_32x32x16_bf16
//   KIND_F32  : f32 x f32 -> fp32            v_mfma_f32_32x32x2_f32 (four per 16 bytes of K and lane)
//
// Naming inside the kernel: P is the operand whose row index runs along the unit-stride
// dimension of D (it is fed as MFMA operand "B", so its index lands on lane%32 of the
// accumulator and stores coalesce); Q is the other one (MFMA operand "A", index on the
// accumulator VGPRs).  For a column-major D, P = op(A) rows (i) and Q = op(B) columns (j); for a
// row-major D the planner sets `swapped` and P/Q trade places.
//
// LDS rows of 128 B are split in eight 16-byte chunks whose position is XOR-swizzled with the row
// number so that both the 1 KiB-per-instruction LDS fills and the ds_read_b128 fragment loads are
// conflict-free (16 consecutive rows reading the same logical chunk hit 16 distinct 16-byte bank
// groups).
#pragma once
#include "numeric.hpp"
#include "store_window.hpp"

namespace zluda_amd {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

enum { KIND_I8 = 0, KIND_F8 = 1, KIND_MXF4 = 2, KIND_F16 = 3, KIND_BF16 = 4, KIND_F32 = 5 };
// 16-bit elements: 16 bytes (8 elements) of K per lane and MFMA, i.e. the byte geometry of int8
constexpr bool kind_is_h16(int kind) { return kind == KIND_F16 || kind == KIND_BF16; }
// bytes per element of the kinds whose elements are whole bytes
constexpr int kind_esz(int kind) { return kind_is_h16(kind) ? 2 : (kind == KIND_F32 ? 4 : 1); }
// f32: a lane's 16 bytes are four K elements, one v_mfma_f32_32x32x2_f32 each; element e of lane group g of the
// 32-byte step s is K index 8 s + 4 g + e for both operands, which is all the instruction asks of a K order

// depends on r mod 32 only, so rows 32 apart (the MFMA tiles of one wave) share a swizzle
__device__ __forceinline__ int swz(int r) { return (r ^ ((r >> 3) & 3)) & 7; }

// Accumulator element -> 32 raw bits.  Takes the element BY VALUE: __builtin_bit_cast applied
// directly to a vector-element expression reads element 0 whatever the index.
__device__ __forceinline__ int to_bits(int x) { return x; }
__device__ __forceinline__ int to_bits(float x) { return (int)f2bits(x); }

template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// 16 bytes per lane from a buffer straight into LDS (buffer_load_dwordx4 ... lds).  `lds_dst` is the
// wave-uniform start of the 1 KiB block the instruction fills; lane l lands at byte l*16.
// The address-space cast only exists in the device pass.
// AUX: the cache policy bits of the instruction (0: default; 2: nt, for bytes that are read once).
template <int AUX = 0>
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t rs, void *lds_dst, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)lds_dst, 16, voff,
                                           soff, 0, AUX);
#endif
}

// 4 bytes per lane from a buffer straight into LDS (buffer_load_dword ... lds): lane l lands at byte l*4 of the 256-byte
// block that starts at the wave-uniform `lds_dst`.
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t rs, void *lds_dst, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)lds_dst, 4, voff, soff, 0, 0);
#endif
}

// 128-bit buffer store whose data registers stay untouched for the wait states that follow it.  Observed on
// MI355X: when the instruction right behind a buffer_store_dwordx4 (offen, scalar offset in an SGPR) is a
// VALU write to the first data register, the store now and then writes the new value instead (element 0 of
// the four, in a few hundred of 131072 outputs); the compiler's hazard table does not list this case, so it
// puts no wait state there.  The asm keeps the data registers live across an s_nop that follows the store.
// AUX: cache policy bits (2 = nt: results that nobody reads back soon; measured on the four-wave kernel's 256 MiB of
// int32 at 8192^3: 392 us instead of 402).
template <int AUX = 0>
__device__ __forceinline__ void buffer_store_b128_guarded(v4i data, __amdgpu_buffer_rsrc_t rs, int voff, int soff) {
  __builtin_amdgcn_raw_buffer_store_b128(data, rs, voff, soff, AUX);
  asm volatile("s_nop 1" : "+v"(data)::"memory");
}

struct MfmaParams {
  GemmArgs g;
  int32_t swapped;           // P = op(B)^T rows, Q = op(A) rows
  int32_t tiles_p, tiles_q;  // tile counts along P and Q
  int32_t group_p;           // raster group height (tiles along P)
  // split-K (splits > 1): workgroup z of gridDim.z handles stages [z * split_stages, ...) of K and
  // writes its raw partial tile to ws[(z * batch + bt)][tiles_q * BQ][tiles_p * BP] (int32 / fp32)
  int32_t splits, split_stages;
  int32_t groups;            // workgroups that walk the tiles (gemm_mfma_short.hpp)
  void *ws;
};

// Workgroup -> tile, batch and share of K.  The hardware hands workgroups to the 8 XCDs, each with an L2 of its own, in turn;
// here every XCD gets a contiguous range of the work, in which the shares of K come outermost, then the batches, then the
// tiles in groups of group_p along P: what its CUs run at one time shares operand panels.  (A range of whole batches: the products
// of a batch read the same operands.  Only a batch whose tiles fill the chip by themselves is spread over all XCDs, so that
// the operands of one batch at a time have to stay in the memory-side cache.)
// Measured (us, before: tiles of a batch over all XCDs, in dispatch order where they are no multiple of 8): bf16 128 x 1000 x 1000, 64
// batches 47.9 -> 43.2; 80 x 351 x 2459, 21 batches 25.1 -> 23.5; MXFP4 1543 x 1530 x 7168, 2 batches 39.1 -> 36.5; int8
// 5000 x 1300 x 1024, 220 tiles 14.6 -> 13.4; bf16 1024 x 512 x 32003 in eight shares 81.8 -> 76.8.
// `id`: position in dispatch order, counted over tiles, then batches, then shares.
struct WorkItem { int p, q, bt, z; };
__device__ __forceinline__ uint32_t lesser(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ WorkItem work_item(const MfmaParams &prm, uint32_t id) {
  const uint32_t tiles = (uint32_t)(prm.tiles_p * prm.tiles_q), batch = (uint32_t)prm.g.batch, n = tiles * batch * (uint32_t)prm.splits;
  const uint32_t x = (id & 7) * (n >> 3) + lesser(id & 7, n & 7) + (id >> 3);
  uint32_t w = x;
  WorkItem it;
  it.bt = it.z = 0;
  // (a branch forward over what only batches and shares need: moved behind the kernel's end, it would return over the whole of it)
  if (n != tiles) {
    const bool by_batch = (tiles & 7) == 0 && tiles >= 256;
    const uint32_t at = by_batch ? id : x, r = at / tiles;
    w = at - r * tiles;
    if (by_batch) w = (w & 7) * (tiles >> 3) + (w >> 3);
    it.z = __builtin_amdgcn_readfirstlane((int)(r / batch));
    it.bt = __builtin_amdgcn_readfirstlane((int)(r % batch));
  }
  const uint32_t group = (uint32_t)(prm.group_p * prm.tiles_q), gid = w / group, first = gid * (uint32_t)prm.group_p;
  const uint32_t in = w - gid * group, rows = lesser((uint32_t)prm.tiles_p - first, (uint32_t)prm.group_p);
  // (divided in vector registers: back to scalar ones, where what is derived from them belongs)
  it.q = __builtin_amdgcn_readfirstlane((int)(in / rows));
  it.p = __builtin_amdgcn_readfirstlane((int)(first + in - (in / rows) * rows));
  return it;
}
// of this workgroup, in a grid of tiles x batches x shares
__device__ __forceinline__ WorkItem work_item(const MfmaParams &prm) {
  const uint32_t tiles = (uint32_t)(prm.tiles_p * prm.tiles_q);
  return work_item(prm, blockIdx.x + tiles * (blockIdx.y + (uint32_t)prm.g.batch * blockIdx.z));
}

// General fused epilogue of the MFMA kernels: any D type, C read, vectors along either dimension,
// partial tiles.  Correct for everything the planner admits, but it spends ~150 instructions per
// four outputs; the fast paths in mfma_store_tile below take the common cases.
// The caller guarantees that every wave of the workgroup has finished reading the LDS tiles (a
// barrier after the K loop); `lds_words` is the start of the workgroup's LDS, reused as staging.
template <int KIND, int WP, int WQ, int WTP, int WTQ, class AccV>
__device__ __forceinline__ void mfma_store_tile_general(const MfmaParams &prm, AccV (&acc)[WTQ / 32][WTP / 32],
                                                int *lds_words, size_t lds_bytes, int p0, int q0, int NP,
                                                int NQ, int bt) {
  constexpr int TP = WTP / 32, TQ = WTQ / 32;
  const GemmArgs &g = prm.g;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wp = wave % WP, wq = wave / WP;
  const int lr = lane & 31, gsel = lane >> 5;
  (void)lds_bytes;
  // ---- epilogue --------------------------------------------------------------------------
  // The accumulators go through LDS (free after the main loop) so that every lane ends up with
  // four consecutive elements along the unit-stride dimension of D: stores are 8 B (bf16) or
  // 16 B (int32/fp32) per lane and contiguous across the 16/32 lanes that share a D column.
  // Each wave stages 16 Q-rows x WTP P-columns per pass in its own LDS region.
  constexpr int SROW = WTP + 8;              // dwords; +8 keeps the two lane halves on distinct banks
  constexpr int LPR = WTP / 4;               // lanes per staged row
  constexpr int RPI = 64 / LPR;              // staged rows read per instruction (96-wide wave tiles: 2, lanes 48-63 idle)
  constexpr int ITER = 16 / RPI;
  static_assert(16 % RPI == 0, "whole passes");
  int *stage = lds_words + wave * (16 * SROW);

  Epilogue ep(g, bt);
  const bool swp = prm.swapped != 0;
  const int pl = (lane % LPR) * 4, qsub = lane / LPR;
  const int pi0 = p0 + wp * WTP + pl;
  // quantities that depend on the P index only: fixed per lane for the whole epilogue
  float p_scale[4], p_bias[4], p_beta[4];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int pi = min(pi0 + e, NP - 1);
    p_scale[e] = g.int_scale ? 1.0f : (swp ? ep.col_scale(pi) : ep.row_scale(pi));
    p_bias[e] = (g.int_scale || swp) ? 0.0f : ep.bias_at(pi);
    p_beta[e] = (g.int_scale || swp) ? 0.0f : ep.beta_at(pi);
  }
  const int64_t d_sp = swp ? g.d_sj : g.d_si, d_sq = swp ? g.d_si : g.d_sj;  // d_sp == 1
  const int64_t c_sp = swp ? g.c_sj : g.c_si, c_sq = swp ? g.c_si : g.c_sj;
  const uint32_t dbits = g.d_type == CUDA_R_32F || g.d_type == CUDA_R_32I ? 32 : g.d_type == CUDA_R_8I ? 8 : 16;
  const bool int_fast = g.int_scale && g.alpha_mode != VECTOR_DEV && g.beta_mode != VECTOR_DEV;
  int32_t ialpha = 1, ibeta = 0;
  if (int_fast) {
    ialpha = g.alpha_mode == SCALAR_VALUE ? g.alpha_val.i : *(const int32_t *)g.alpha_ptr;
    ibeta = g.beta_mode == SCALAR_VALUE ? g.beta_val.i : *(const int32_t *)g.beta_ptr;
  }

  // `pass` must be a compile-time constant: a rolled loop here would index the accumulator
  // registers dynamically and push them to scratch for the whole kernel.
  auto do_pass = [&](auto pass_c) {
    constexpr int pass = decltype(pass_c)::value;
    constexpr int a = pass >> 1, h = pass & 1;
#pragma unroll
    for (int b = 0; b < TP; b++)
#pragma unroll
      for (int vv = 0; vv < 8; vv++) {
        const int ql = 8 * (vv >> 2) + 4 * gsel + (vv & 3);
        stage[ql * SROW + b * 32 + lr] = to_bits(acc[a][b][h * 8 + vv]);
      }
    __syncthreads();
#pragma unroll 1
    for (int it = 0; it < ITER; it++) {
      const int ql = it * RPI + qsub;
      const int qi = q0 + wq * WTQ + a * 32 + h * 16 + ql;
      const v4i raw = *(const v4i *)&stage[ql * SROW + pl];
      if (qi >= NQ || pi0 >= NP || qsub >= RPI) continue;
      const int64_t dbase = g.d_sb * bt + (int64_t)pi0 * d_sp + (int64_t)qi * d_sq;
      const int64_t cbase = g.c_sb * bt + (int64_t)pi0 * c_sp + (int64_t)qi * c_sq;
      const bool full4 = pi0 + 3 < NP && ((dbase * dbits / 8) & (dbits / 2 - 1)) == 0 &&
                         (((uintptr_t)g.D) & 15) == 0;
      if (g.int_scale) {
        if (int_fast) {
          v4i r;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            uint32_t x = (uint32_t)ialpha * (uint32_t)raw[e];
            if (ibeta != 0 && pi0 + e < NP) x += (uint32_t)ibeta * (uint32_t)((const int32_t *)g.C)[cbase + e * c_sp];
            r[e] = (int)x;
          }
          if (full4) *(v4i *)((int32_t *)g.D + dbase) = r;
          else
#pragma unroll
            for (int e = 0; e < 4; e++) if (pi0 + e < NP) ((int32_t *)g.D)[dbase + e] = r[e];
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (pi0 + e < NP) ep.store_int(swp ? qi : pi0 + e, swp ? pi0 + e : qi, raw[e]);
        }
        continue;
      }
      const float q_scale = swp ? ep.row_scale(qi) : ep.col_scale(qi);
      const float q_bias = swp ? ep.bias_at(qi) : 0.0f;
      const float q_beta = swp ? ep.beta_at(qi) : 0.0f;
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int rawe = raw[e];
        const float accf = KIND == KIND_I8 ? (float)rawe : bits2f((uint32_t)rawe);
        float y = (swp ? q_scale * p_scale[e] : p_scale[e] * q_scale) * accf;
        const float be = swp ? q_beta : p_beta[e];
        if (be != 0.0f && pi0 + e < NP) y += be * ep.sc * load_elem(g.C, g.c_type, cbase + e * c_sp);
        y += swp ? q_bias : p_bias[e];
        x[e] = ep.finish(y);
      }
      if (full4 && dbits == 32 && g.d_type == CUDA_R_32F) {
        *(float4 *)((float *)g.D + dbase) = make_float4(x[0], x[1], x[2], x[3]);
      } else if (full4 && g.d_type == CUDA_R_16BF) {
        uint2 pk;
        pk.x = (uint32_t)enc_bf16(x[0]) | ((uint32_t)enc_bf16(x[1]) << 16);
        pk.y = (uint32_t)enc_bf16(x[2]) | ((uint32_t)enc_bf16(x[3]) << 16);
        *(uint2 *)((uint16_t *)g.D + dbase) = pk;
      } else if (full4 && g.d_type == CUDA_R_16F) {
        uint2 pk;
        pk.x = (uint32_t)enc_f16(x[0]) | ((uint32_t)enc_f16(x[1]) << 16);
        pk.y = (uint32_t)enc_f16(x[2]) | ((uint32_t)enc_f16(x[3]) << 16);
        *(uint2 *)((uint16_t *)g.D + dbase) = pk;
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (pi0 + e < NP) store_elem(g.D, g.d_type, dbase + e, x[e]);
      }
    }
    __syncthreads();
  };
  static_for<TQ * 2>(do_pass);
}

// The kernel's arguments lie in host memory: a cache line of them that a scalar load asks for first costs most of a
// microsecond.  Asked for where they are used, in batches, the lines come one after the other; here all of them are asked for
// together at the kernel's entry (one dword of each), and what is read later comes out of the scalar cache.
__device__ __forceinline__ void fetch_args(const MfmaParams &prm) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int LINES = (sizeof(MfmaParams) + 63) / 64;
  static_assert(LINES == 6, "one operand per line below");
  const uint32_t *w = (const uint32_t *)&prm;
  asm volatile("" ::"s"(w[0]), "s"(w[16]), "s"(w[32]), "s"(w[48]), "s"(w[64]), "s"(w[80]));
#endif
}

// The arguments once more, for what runs behind the K loop.  Read through `prm` the compiler keeps everything an epilogue may
// ask for from the kernel's entry on, has no scalar registers for it and spills.
__device__ __forceinline__ const MfmaParams &args_again(const MfmaParams &prm) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef const __attribute__((address_space(4))) MfmaParams *arg_ptr;
  uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();  // (the kernels' one argument lies at its start)
  asm volatile("" : "+s"(at));
  const MfmaParams &again = *(const MfmaParams *)(arg_ptr)at;
  // (what every float epilogue asks for, in one go: left to its first uses it is a chain of loads and branches)
  const GemmArgs &g = again.g;
  asm volatile("" ::"s"(g.alpha_mode), "s"(g.alpha_val.i), "s"(g.alpha_ptr), "s"(g.a_scale_mode), "s"(g.b_scale_mode), "s"(g.a_scale),
               "s"(g.b_scale), "s"(g.d_scale), "s"(g.bias), "s"(g.bias_type), "s"(g.D), "s"(g.d_sb));
  return again;
#else
  return prm;
#endif
}

// Fast path 1: pure integer epilogue with alpha, beta scalars and beta == 0: D = alpha * acc straight from the accumulator
// registers.  Lanes 0..31 of a store hold 32 consecutive int32 of one D column (one 128-byte line), so no LDS staging is
// needed; two instructions per output element.  Tiles that hang over the end of P (EDGE) mask their lanes, columns past the
// end fall outside the window.
template <int WP, int WQ, int WTP, int WTQ, bool EDGE>
__device__ __forceinline__ void mfma_store_tile_i32(const MfmaParams &prm, v16i (&acc)[WTQ / 32][WTP / 32],
                                                    int p0, int q0, int NP, int NQ, int bt, int ialpha) {
  constexpr int TP = WTP / 32, TQ = WTQ / 32;
  const GemmArgs &g = prm.g;
  // the wave index is uniform by construction; say so, or the buffer descriptor built from it is
  // treated as divergent and every store is wrapped in a readfirstlane loop
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave % WP, wq = wave / WP;
  const int lr = lane & 31, gsel = lane >> 5;
  const int d_sq = (int)(prm.swapped ? g.d_si : g.d_sj);  // < kNarrowPitch (checked by the dispatcher)
  // Buffer stores: wave-uniform descriptor at the wave tile, per-lane byte offset of (row 4*gsel,
  // column lr) in a VGPR, everything else in the scalar offset.
  const int64_t corner = (int64_t)(q0 + wq * WTQ) * d_sq + (p0 + wp * WTP);
  int32_t *Dw = (int32_t *)g.D + g.d_sb * bt + corner;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dw, 0, tile_window_bytes(d_sq, NP, NQ, corner, 4), 0x00020000);
  int voff[TP];
#pragma unroll
  for (int b = 0; b < TP; b++) voff[b] = !EDGE || p0 + wp * WTP + b * 32 + lr < NP ? (4 * gsel * d_sq + lr) * 4 : kStoreNowhere;
  // alpha == 1 (the usual case) stores the accumulator registers as they are
  if (ialpha == 1) {
#pragma unroll
    for (int a = 0; a < TQ; a++)
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int soff = (a * 32 + 8 * (v >> 2) + (v & 3)) * d_sq * 4;  // uniform
#pragma unroll
        for (int b = 0; b < TP; b++) __builtin_amdgcn_raw_buffer_store_b32(acc[a][b][v], rs, voff[b], soff + b * 128, 0);
      }
  } else {
#pragma unroll
    for (int a = 0; a < TQ; a++)
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int soff = (a * 32 + 8 * (v >> 2) + (v & 3)) * d_sq * 4;
#pragma unroll
        for (int b = 0; b < TP; b++)
          __builtin_amdgcn_raw_buffer_store_b32(acc[a][b][v] * ialpha, rs, voff[b], soff + b * 128, 0);
      }
  }
}

// Split-K partial tile: the raw accumulators (int32, or fp32 bit patterns) of a whole tile into the
// padded workspace matrix of pitch `ws_pitch` dwords; same store pattern as mfma_store_tile_i32.
template <int WP, int WQ, int WTP, int WTQ, class AccV>
__device__ __forceinline__ void mfma_store_tile_raw(int32_t *ws_tile, int ws_pitch, AccV (&acc)[WTQ / 32][WTP / 32]) {
  constexpr int TP = WTP / 32, TQ = WTQ / 32;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave % WP, wq = wave / WP;
  const int lr = lane & 31, gsel = lane >> 5;
  int32_t *Dw = ws_tile + (int64_t)(wq * WTQ) * ws_pitch + wp * WTP;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dw, 0, 0xFFFFFFFF, 0x00020000);
  const int voff = (4 * gsel * ws_pitch + lr) * 4;
#pragma unroll
  for (int a = 0; a < TQ; a++)
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int soff = (a * 32 + 8 * (v >> 2) + (v & 3)) * ws_pitch * 4;  // uniform
#pragma unroll
      for (int b = 0; b < TP; b++) __builtin_amdgcn_raw_buffer_store_b32(to_bits(acc[a][b][v]), rs, voff, soff + b * 128, 0);
    }
}

// Fast path 2, for what fast path 3 does not take: float epilogue without a C read (beta == 0), D of type bf16, f16 or f32 at
// any element's address and any pitch, straight from the accumulator registers.  One 32 x 32 tile (16 accumulators per lane) at a time: the activation and
// the type of D are uniform branches around whole tiles, so one body serves every combination.
// f32: lanes 0..31 of a store hold 32 consecutive elements of one D column.  16-bit types: lane (lr, gsel) holds element
// (column lr, row 8*(v/4)+4*gsel+v%4); rows 2k and 2k+1 are paired: after one DPP swap with the neighbouring lane the even
// lane owns columns (lr, lr+1) of row 2k and the odd lane columns (lr-1, lr) of row 2k+1, so every lane stores one dword of
// two results and a store instruction writes four 64-byte row segments.  (The memory system takes those dwords at 2-byte
// alignment as well: an odd pitch of D costs nothing here.)
// A tile that hangs over the end of P (EDGE) masks its lanes; the pair that straddles an odd end is stored as one 16-bit element.
// Measured (MI355X, us, before: the element-wise path through LDS on every tile that was not whole or not 16-byte aligned):
// bf16 1000 x 1000 x 128, 64 batches, with the product that follows it 286 -> 146; int8 -> int32 5004 x 3000 x 4096 110 -> 61;
// bf16 5001 x 4099 x 4096 + bias + GELU 258 -> 186.
template <int KIND, int WP, int WQ, int WTP, int WTQ, bool EDGE, class AccV>
__device__ __forceinline__ void mfma_store_tile_float(const MfmaParams &prm, AccV (&acc)[WTQ / 32][WTP / 32],
                                                      int p0, int q0, int NP, int NQ, int bt) {
  constexpr int TP = WTP / 32, TQ = WTQ / 32;
  const GemmArgs &g = prm.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave % WP, wq = wave / WP;
  const int lr = lane & 31, gsel = lane >> 5, odd = lane & 1;
  Epilogue ep(g, bt);
  const bool swp = prm.swapped != 0;
  const bool to_f32 = g.d_type == CUDA_R_32F, to_bf16 = g.d_type == CUDA_R_16BF;
  const int esz = to_f32 ? 4 : 2;
  const int pc = p0 + wp * WTP, qc = q0 + wq * WTQ;
  // vectors that run along Q (per-column scale, or per-row quantities of a row-major D)
  const bool q_vec = swp ? (ep.alpha_v || ep.sa_v || g.bias) : (ep.sb_v != nullptr);
  const float q_scale = swp ? ep.row_scale(0) : ep.col_scale(0);  // used when !q_vec
  float p_scale[TP], p_bias[TP];
#pragma unroll
  for (int b = 0; b < TP; b++) {
    const int pi = EDGE ? min(pc + b * 32 + lr, NP - 1) : pc + b * 32 + lr;
    p_scale[b] = swp ? ep.col_scale(pi) : ep.row_scale(pi);
    p_bias[b] = swp ? 0.0f : ep.bias_at(pi);
    if (!q_vec) p_scale[b] *= q_scale;
  }
  // the vectors along Q, lane l holding entry l % 32 of each 32 columns (one burst of loads up front: a load per column
  // where it is used costs a memory round trip per 32 columns -- 4096 x 777 x 14336 int8 with per-token scales 92 us against 88)
  float q_lane[TQ], qb_lane[TQ];
#pragma unroll
  for (int a = 0; a < TQ; a++) {
    const int qi = min(qc + a * 32 + lr, NQ - 1);  // columns past the end: dropped stores
    q_lane[a] = q_vec ? (swp ? ep.row_scale(qi) : ep.col_scale(qi)) : 1.0f;
    qb_lane[a] = q_vec && swp ? ep.bias_at(qi) : 0.0f;
  }
  const int d_sq = (int)(swp ? g.d_si : g.d_sj);  // < kNarrowPitch (checked by the dispatcher)
  const int64_t corner = (int64_t)qc * d_sq + pc;
  char *Dw = (char *)g.D + (g.d_sb * bt + corner) * esz;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dw, 0, tile_window_bytes(d_sq, NP, NQ, corner, esz), 0x00020000);
  const int voff_in = to_f32 ? (4 * gsel * d_sq + lr) * 4 : ((4 * gsel + odd) * d_sq + (lr & ~1)) * 2;
  const bool odd_end = EDGE && (NP & 1) && NP < pc + WTP;  // (uniform) some pair of the wave tile straddles the end

#pragma unroll
  for (int a = 0; a < TQ; a++) {
    float qs[16], qb[16];
#pragma unroll
    for (int v = 0; v < 16; v++) { qs[v] = 1.0f; qb[v] = 0.0f; }
    if (q_vec) {
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int from = (8 * (v >> 2) + 4 * gsel + (v & 3)) * 4;  // the lane that holds the column, in bytes
        qs[v] = bits2f((uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)f2bits(q_lane[a])));
        if (swp) qb[v] = bits2f((uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)f2bits(qb_lane[a])));
      }
    }
#pragma unroll
    for (int b = 0; b < TP; b++) {
      float x[16];
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const float accf = KIND == KIND_I8 ? (float)to_bits(acc[a][b][v]) : bits2f((uint32_t)to_bits(acc[a][b][v]));
        x[v] = accf;
      }
      if (q_vec) {
#pragma unroll
        for (int v = 0; v < 16; v++) x[v] = (p_scale[b] * qs[v]) * x[v] + (p_bias[b] + qb[v]);
      } else {
#pragma unroll
        for (int v = 0; v < 16; v++) x[v] = p_scale[b] * x[v] + p_bias[b];
      }
      if (g.act == ACT_GELU) {
#pragma unroll
        for (int v = 0; v < 16; v++) x[v] = gelu_tanh(x[v]);
      } else if (g.act == ACT_RELU) {
#pragma unroll
        for (int v = 0; v < 16; v++) x[v] = x[v] > 0.0f ? x[v] : 0.0f;
      }
#pragma unroll
      for (int v = 0; v < 16; v++) x[v] *= ep.sd;
      const int tile_p = pc + b * 32;
      const int voff = !EDGE || tile_p + (to_f32 ? lr : lr | 1) < NP ? voff_in : kStoreNowhere;
      if (to_f32) {
#pragma unroll
        for (int v = 0; v < 16; v++)
          __builtin_amdgcn_raw_buffer_store_b32((int)f2bits(x[v]), rs, voff, (a * 32 + 8 * (v >> 2) + (v & 3)) * d_sq * 4 + b * 128, 0);
      } else {
        uint32_t pk[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
          // even lanes keep row 2k and need the neighbour's row-2k value; odd lanes the other way round
          const float mine = odd ? x[2 * k + 1] : x[2 * k], give = odd ? x[2 * k] : x[2 * k + 1];
          const float got = bits2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2bits(give), 0xB1 /* quad_perm [1,0,3,2] */, 0xF, 0xF, true));
          x[2 * k] = odd ? got : mine;
          x[2 * k + 1] = odd ? mine : got;
        }
        if (to_bf16) {
#pragma unroll
          for (int k = 0; k < 8; k++) pk[k] = pack_bf16x2(x[2 * k], x[2 * k + 1]);
        } else {
#pragma unroll
          for (int k = 0; k < 8; k++) pk[k] = pack_f16x2(x[2 * k], x[2 * k + 1]);
        }
#pragma unroll
        for (int k = 0; k < 8; k++)
          __builtin_amdgcn_raw_buffer_store_b32((int)pk[k], rs, voff, (a * 32 + 8 * (k >> 1) + 2 * (k & 1)) * d_sq * 2 + b * 64, 0);
        if (odd_end) {
          const int vedge = tile_p + (lr & ~1) == NP - 1 ? voff_in : kStoreNowhere;
#pragma unroll
          for (int k = 0; k < 8; k++)
            __builtin_amdgcn_raw_buffer_store_b16((short)pk[k], rs, vedge, (a * 32 + 8 * (k >> 1) + 2 * (k & 1)) * d_sq * 2 + b * 64, 0);
        }
      }
    }
  }
}

// Fast path 3: the same for whole tiles where nothing varies along Q, which is most of what runs here.  The activation and
// the type (DT: 0 bf16, 1 f16, 2 f32) are fixed at compile time and the tiles of a row are walked together: the stores start
// with the first values, are spread over the arithmetic, and those of neighbouring tiles (for 16-bit types the two halves of
// a cache line) follow each other.  Measured (MI355X, us, fast path 2 on the same tiles -> this): 4096 x 2048 x 256 fp8 -> bf16
// 10.7 -> 9.4, bf16 -> bf16 12.8 -> 11.3, fp8 -> f32 12.3 -> 11.3; 2048 x 2048 x 1024 int8 -> bf16 10.7 -> 9.5.  (Holding a row of
// tiles and storing it at the end: 13.5 instead of 11.3, the stores then wait for all of the arithmetic.)
template <int KIND, int WP, int WQ, int WTP, int WTQ, int ACT, int DT, class AccV>
__device__ __forceinline__ void mfma_store_tile_plain(const MfmaParams &prm, AccV (&acc)[WTQ / 32][WTP / 32], int p0, int q0, int NP,
                                                      int NQ, int bt) {
  constexpr int TP = WTP / 32, TQ = WTQ / 32, ESZ = DT == 2 ? 4 : 2;
  const GemmArgs &g = prm.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave % WP, wq = wave / WP;
  const int lr = lane & 31, gsel = lane >> 5, odd = lane & 1;
  Epilogue ep(g, bt);
  const bool swp = prm.swapped != 0;
  const int pc = p0 + wp * WTP, qc = q0 + wq * WTQ;
  const float q_scale = swp ? ep.row_scale(0) : ep.col_scale(0);
  float p_scale[TP], p_bias[TP];
#pragma unroll
  for (int b = 0; b < TP; b++) {
    const int pi = pc + b * 32 + lr;
    p_scale[b] = (swp ? ep.col_scale(pi) : ep.row_scale(pi)) * q_scale;
    p_bias[b] = swp ? 0.0f : ep.bias_at(pi);
  }
  const int d_sq = (int)(swp ? g.d_si : g.d_sj);  // < kNarrowPitch (checked by the dispatcher)
  const int64_t corner = (int64_t)qc * d_sq + pc;
  char *Dw = (char *)g.D + (g.d_sb * bt + corner) * ESZ;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dw, 0, tile_window_bytes(d_sq, NP, NQ, corner, ESZ), 0x00020000);
  const int voff = DT == 2 ? (4 * gsel * d_sq + lr) * 4 : ((4 * gsel + odd) * d_sq + (lr & ~1)) * 2;
  auto value = [&](int raw, int b) {
    float y = p_scale[b] * (KIND == KIND_I8 ? (float)raw : bits2f((uint32_t)raw)) + p_bias[b];
    if (ACT == ACT_RELU) y = y > 0.0f ? y : 0.0f;
    else if (ACT == ACT_GELU) y = gelu_tanh(y);
    return y * ep.sd;
  };
#pragma unroll
  for (int a = 0; a < TQ; a++)
#pragma unroll
    for (int k = 0; k < 8; k++) {  // rows 2k and 2k + 1 of tile a's lanes
      const int soff = (a * 32 + 8 * (k >> 1) + 2 * (k & 1)) * d_sq * ESZ;  // uniform
      if constexpr (DT == 2) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
          for (int b = 0; b < TP; b++)
            __builtin_amdgcn_raw_buffer_store_b32((int)f2bits(value(to_bits(acc[a][b][2 * k + r]), b)), rs, voff, soff + r * d_sq * 4 + b * 128, 0);
      } else {
#pragma unroll
        for (int b = 0; b < TP; b++) {
          const float x0 = value(to_bits(acc[a][b][2 * k]), b), x1 = value(to_bits(acc[a][b][2 * k + 1]), b);
          // even lanes keep row 2k and need the neighbour's row-2k value; odd lanes the other way round
          const float mine = odd ? x1 : x0, give = odd ? x0 : x1;
          const float got = bits2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2bits(give), 0xB1 /* quad_perm [1,0,3,2] */, 0xF, 0xF, true));
          const float lo = odd ? got : mine, hi = odd ? mine : got;
          __builtin_amdgcn_raw_buffer_store_b32((int)(DT == 0 ? pack_bf16x2(lo, hi) : pack_f16x2(lo, hi)), rs, voff, soff + b * 64, 0);
        }
      }
    }
}

// What the epilogues with an aux matrix read it from, write it to, and put D and the partial sums of its rows
// (DGELU_BGRAD) into; one column of a wave's tile is `q` elements of that pitch further on.
// The fused forms take 16-bit floats, a column-major D, beta == 0, one factor for all of D, a multiple of 8 rows and 16-byte aligned
// columns of D and aux (aux_in_epilogue() of the launch layer); everything else has a pass of its own behind the matmul (aux_epilogue.hpp).
struct AuxTile {
  __amdgpu_buffer_rsrc_t rs_d, rs_x;
  int d_sq, x_sq;
  float factor;
  float *sums;  // this wave's partial sums, indexed by P; or NULL
  __device__ __forceinline__ AuxTile(const MfmaParams &prm, const EpilogueScalars &s, int pc, int qc, int NP, int NQ, int bt, int share, int shares) {
    const GemmArgs &g = prm.g;
    d_sq = (int)g.d_sj; x_sq = (int)g.aux_sj;  // < kNarrowPitch
    const int64_t d_corner = (int64_t)qc * d_sq + pc, x_corner = (int64_t)qc * x_sq + pc;
    rs_d = __builtin_amdgcn_make_buffer_rsrc((char *)g.D + (g.d_sb * bt + d_corner) * 2, 0, tile_window_bytes(d_sq, NP, NQ, d_corner, 2), 0x00020000);
    rs_x = __builtin_amdgcn_make_buffer_rsrc((char *)g.aux + (g.aux_sb * bt + x_corner) * 2, 0, tile_window_bytes(x_sq, NP, NQ, x_corner, 2), 0x00020000);
    factor = s.alpha_s * s.sa_s * s.sb_s;
    sums = g.aux_bgrad ? (float *)prm.ws + ((int64_t)bt * shares + share) * NP : nullptr;
  }
};

// The two 16-bit floats of a dword, and back
__device__ __forceinline__ float low_half(uint32_t d, bool bf16) { return bf16 ? bits2f(d << 16) : dec_f16((uint16_t)d); }
__device__ __forceinline__ float high_half(uint32_t d, bool bf16) { return bf16 ? bits2f(d & 0xffff0000u) : dec_f16((uint16_t)(d >> 16)); }
__device__ __forceinline__ uint32_t pack_halves(float lo, float hi, bool bf16) { return bf16 ? pack_bf16x2(lo, hi) : pack_f16x2(lo, hi); }

// GELU with its input kept (MODE 1: aux = x, D = gelu(x)) and its gradient (MODE 2: D = x * gelu'(aux), and the sums of this
// wave's part of D's rows): aux goes through the same dwords as D (fast path 2), one 32 x 32 tile at a time.
template <int WP, int WQ, int WTP, int WTQ, int MODE, class AccV>
__device__ __forceinline__ void mfma_store_tile_aux(const MfmaParams &prm, AccV (&acc)[WTQ / 32][WTP / 32], int p0, int q0, int NP, int NQ, int bt) {
  constexpr int TP = WTP / 32, TQ = WTQ / 32;
  const GemmArgs &g = prm.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave % WP, wq = wave / WP;
  const int lr = lane & 31, gsel = lane >> 5, odd = lane & 1;
  const int pc = p0 + wp * WTP, qc = q0 + wq * WTQ;
  const Epilogue ep(g, bt);
  const AuxTile at(prm, EpilogueScalars(g), pc, qc, NP, NQ, bt, q0 / WTQ + wq, prm.tiles_q * WQ);
  const bool bf16 = g.d_type == CUDA_R_16BF;
  const int vd = ((4 * gsel + odd) * at.d_sq + (lr & ~1)) * 2, vx = ((4 * gsel + odd) * at.x_sq + (lr & ~1)) * 2;
  float p_bias[TP], sum[TP][2];
#pragma unroll
  for (int b = 0; b < TP; b++) {
    p_bias[b] = MODE == 1 ? ep.bias_at(min(pc + b * 32 + lr, NP - 1)) : 0.0f;
    sum[b][0] = sum[b][1] = 0.0f;
  }
#pragma unroll
  for (int a = 0; a < TQ; a++) {
    // (the row's aux dwords in one burst)
    uint32_t x_in[TP][8];
    if constexpr (MODE == 2) {
#pragma unroll
      for (int b = 0; b < TP; b++)
#pragma unroll
        for (int k = 0; k < 8; k++)
          x_in[b][k] = __builtin_amdgcn_raw_buffer_load_b32(at.rs_x, pc + b * 32 + lr < NP ? vx : kStoreNowhere, (a * 32 + 8 * (k >> 1) + 2 * (k & 1)) * at.x_sq * 2 + b * 64, 0);
    }
#pragma unroll
    for (int b = 0; b < TP; b++) {
      const bool in = pc + b * 32 + lr < NP;  // (a pair never straddles the end: it is a multiple of 8)
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const float x0 = at.factor * bits2f((uint32_t)to_bits(acc[a][b][2 * k])) + p_bias[b];
        const float x1 = at.factor * bits2f((uint32_t)to_bits(acc[a][b][2 * k + 1])) + p_bias[b];
        // even lanes keep row 2k and need the neighbour's row-2k value; odd lanes the other way round
        const float mine = odd ? x1 : x0, give = odd ? x0 : x1;
        const float got = bits2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2bits(give), 0xB1 /* quad_perm [1,0,3,2] */, 0xF, 0xF, true));
        float lo = odd ? got : mine, hi = odd ? mine : got;
        const int row = a * 32 + 8 * (k >> 1) + 2 * (k & 1);
        if constexpr (MODE == 1) {
          __builtin_amdgcn_raw_buffer_store_b32((int)pack_halves(lo, hi, bf16), at.rs_x, in ? vx : kStoreNowhere, row * at.x_sq * 2 + b * 64, 0);
          lo = gelu_tanh(lo) * ep.sd;
          hi = gelu_tanh(hi) * ep.sd;
        } else {
          lo *= dgelu_tanh(low_half(x_in[b][k], bf16));
          hi *= dgelu_tanh(high_half(x_in[b][k], bf16));
          // (columns past the end hold products of some column)
          const bool counts = qc + row + 4 * gsel + odd < NQ;
          sum[b][0] += counts ? lo : 0.0f;
          sum[b][1] += counts ? hi : 0.0f;
        }
        __builtin_amdgcn_raw_buffer_store_b32((int)pack_halves(lo, hi, bf16), at.rs_d, in ? vd : kStoreNowhere, row * at.d_sq * 2 + b * 64, 0);
      }
      __builtin_amdgcn_sched_barrier(0);  // one tile at a time: what the scheduler hoists across them spills
    }
  }
  if (MODE == 2 && at.sums) {
#pragma unroll
    for (int b = 0; b < TP; b++) {
#pragma unroll
      for (int e = 0; e < 2; e++) {  // over the even and the odd lane of a pair of columns, and the lane halves
        sum[b][e] += __shfl_xor(sum[b][e], 1, 64);
        sum[b][e] += __shfl_xor(sum[b][e], 32, 64);
      }
      const int p = pc + b * 32 + lr;
      if (gsel == 0 && p < NP) at.sums[p] = sum[b][odd];
    }
  }
}

// Epilogue dispatch: the fast paths for the common configurations, the general path for the rest (C reads, 8-bit outputs,
// integer outputs of a float epilogue, vectors of alpha in the integer one).  All conditions are workgroup-uniform.  What they
// and the integer path read is few enough to be kept from the kernel's entry on; the float paths read the arguments again.
// AUX: kernels of their own carry the epilogues with an aux matrix, and nothing else (as one more branch here they cost plain products of
// one or two rounds 0.3 us: bf16 777 x 512 x 64, 64 batches 22.3 -> 22.7, 2048 x 2176 x 704 A:N B:T 15.0 -> 15.4).
template <int KIND, int WP, int WQ, int WTP, int WTQ, bool AUX, class AccV>
__device__ __forceinline__ void mfma_store_tile(const MfmaParams &prm, AccV (&acc)[WTQ / 32][WTP / 32],
                                                int *lds_words, size_t lds_bytes, int p0, int q0, int NP,
                                                int NQ, int bt) {
  const GemmArgs &g = prm.g;
  if constexpr (AUX) {
    static_assert(kind_is_h16(KIND) && aux_on_wave_tile32(WTP, WTQ), "aux_in_epilogue()");
    const MfmaParams &late = args_again(prm);
    if (g.act == ACT_GELU_KEPT) mfma_store_tile_aux<WP, WQ, WTP, WTQ, 1>(late, acc, p0, q0, NP, NQ, bt);
    else mfma_store_tile_aux<WP, WQ, WTP, WTQ, 2>(late, acc, p0, q0, NP, NQ, bt);
    return;
  }
  const int64_t d_sq = prm.swapped ? g.d_si : g.d_sj;
  const bool narrow = d_sq < kNarrowPitch;  // the lane offsets fit 32 bits
  const bool whole = p0 + WP * WTP <= NP;
  if constexpr (KIND == KIND_I8) {
    if (g.int_scale && narrow && g.alpha_mode != VECTOR_DEV && g.beta_mode == SCALAR_VALUE && g.beta_val.i == 0) {
      const int ialpha = g.alpha_mode == SCALAR_VALUE ? g.alpha_val.i : *(const int32_t *)g.alpha_ptr;
      if (whole) mfma_store_tile_i32<WP, WQ, WTP, WTQ, false>(prm, acc, p0, q0, NP, NQ, bt, ialpha);
      else mfma_store_tile_i32<WP, WQ, WTP, WTQ, true>(prm, acc, p0, q0, NP, NQ, bt, ialpha);
      return;
    }
  }
  const MfmaParams &late = args_again(prm);
  if (!g.int_scale && narrow && g.beta_mode == SCALAR_VALUE && g.beta_val.f == 0.0f &&
      (g.d_type == CUDA_R_16BF || g.d_type == CUDA_R_16F || g.d_type == CUDA_R_32F)) {
    if (!whole) {
      mfma_store_tile_float<KIND, WP, WQ, WTP, WTQ, true>(late, acc, p0, q0, NP, NQ, bt);
      return;
    }
    // what varies along Q: a scale vector of B's, or a row-major D's per-row quantities
    const bool q_vec = prm.swapped ? g.alpha_mode == VECTOR_DEV || late.g.a_scale_mode == SCALE_OUTER_VEC || late.g.bias != nullptr
                                   : late.g.b_scale_mode == SCALE_OUTER_VEC;
    if (q_vec) {
      mfma_store_tile_float<KIND, WP, WQ, WTP, WTQ, false>(late, acc, p0, q0, NP, NQ, bt);
      return;
    }
#define ZLUDA_EPI_PLAIN(ACT_, DT_) mfma_store_tile_plain<KIND, WP, WQ, WTP, WTQ, ACT_, DT_>(late, acc, p0, q0, NP, NQ, bt)
#define ZLUDA_EPI_ACT(DT_)                                  \
  if (g.act == ACT_GELU) ZLUDA_EPI_PLAIN(ACT_GELU, DT_);    \
  else if (g.act == ACT_RELU) ZLUDA_EPI_PLAIN(ACT_RELU, DT_); \
  else ZLUDA_EPI_PLAIN(ACT_NONE, DT_);
    if (g.d_type == CUDA_R_16BF) {
      ZLUDA_EPI_ACT(0)
    } else if (g.d_type == CUDA_R_16F) {
      ZLUDA_EPI_ACT(1)
    } else {
      ZLUDA_EPI_ACT(2)
    }
#undef ZLUDA_EPI_ACT
#undef ZLUDA_EPI_PLAIN
    return;
  }
  mfma_store_tile_general<KIND, WP, WQ, WTP, WTQ>(late, acc, lds_words, lds_bytes, p0, q0, NP, NQ, bt);
}

} // namespace zluda_amd
