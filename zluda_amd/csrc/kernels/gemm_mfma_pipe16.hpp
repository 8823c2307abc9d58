// MFMA GEMM for K-contiguous int8 / fp8 operands on gfx950 built on the 16x16 instruction shapes
//   int8 : v_mfma_i32_16x16x64_i8            fp8 : v_mfma_f32_16x16x128_f8f6f4
// inside the K loop of gemm_mfma_pipe.hpp (LDS ring filled by buffer_load ... lds in whole 128-byte row
// segments, XOR-swizzled 16-byte chunks, XCD-aware workgroup -> tile order, one barrier per stage, split-K
// through the workspace).
//
// Why a second MFMA shape: the part is power limited under matrix load, so a large GEMM takes as long as
// its energy allows, and the 16x16 shapes need less of it.  Measured on MI355X at its 1400 W cap (8192^3,
// kernels running back to back for seconds, board power read from hwmon): with nothing changed but the
// instruction, the 256 x 256 tile kernel takes 5 % less time for fp8 and 7 % less for int8.  The 16x16
// shapes reduce over a deeper K per instruction and touch the accumulators half as often per multiply-add.
//
// What differs from gemm_mfma_pipe.hpp:
//   * P is the MFMA operand "A": the 16x16 result layout then gives every lane FOUR CONSECUTIVE elements
//     along D's unit-stride dimension (rows 4*(lane/16) .. +3 of a 16-row tile, column lane%16), so the
//     epilogue stores 16 bytes per lane straight from the accumulators (bf16 / f16: the 8 bytes of two tiles, traded
//     between neighbouring lane groups): no LDS staging.
//   * A fragment is 16 rows x 128 K bytes: lane l holds row l%16 and the K bytes of lane group l/16 --
//     fp8: chunks 2*(l/16) and 2*(l/16)+1 of the 128-byte row (one instruction per stage and tile pair);
//     int8 and 16-bit: the same two chunks, one for each of two instructions.  Both operands use the same assignment,
//     which is all a dot product needs.  (A ds_read_b128 is served in four parts, the lanes {0-3, 12-15, 20-23, 24-27},
//     {4-7, 8-11, 16-19, 28-31} and the same of the upper half: two lane groups in each, whose chunks have to be two apart
//     for the swizzle to keep them on different banks.  With the chunks l/16 and 4 + l/16 every read took twice its time; the loops
//     wait for other things more: bf16 4096^3 111.6 -> 109.9 us, 8192^3 775 -> 772, int8 8192^3 413 -> 411.)
//   * A stage is walked in four sub-steps over (P half, Q half) of the wave tile in snake order, so that
//     consecutive sub-steps share one half and only the other is fetched:
//         even stages: (P0,Q0) (P0,Q1) | (P1,Q1) (P1,Q0)        odd stages: (P0,Q1) (P0,Q0) | (P1,Q0) (P1,Q1)
//     Every fragment of the stage has been requested when its second sub-step ends; the barrier sits
//     there ("|"), and behind it the slot is refilled with stage kt+2 while the last two sub-steps fetch
//     the first fragments of stage kt+1 from the other slot into the registers that have just become free.
//     The fragment registers (both P halves, both Q halves) are as many as in gemm_mfma_pipe.hpp.
//
// 16-bit operands with unit stride along their row index ("MC": PMC / QMC; D^T and the gradients of a training step) go
// through the same loop: the DMA copies 64 K rows of 128 or 256 elements as they lie in memory, and ds_read_b64_tr_b16
// (16 lanes read 4 K rows x 16 elements; lane i gets the four K elements of row i) transposes on the way into the
// fragments, so there is no work in registers and no store to LDS.  The kernel of gemm_mfma_tr.hpp, which transposes in
// registers, spends its stages on that: bf16 8192^3 A:N B:N 1019 us there, 808 here; 4096^3 A:N B:N 110; 128 x 128 tiles,
// 2048 x 4096 x 8192 A:N B:N 183 and 133 inside a training step.  (The 128 x 128 tile also has a ring of four stages, see mfma_tr_launch.hpp.)
// LDS layout of such an operand: blocks of 1 KiB, one DMA instruction of a wave each, at a pitch of 1056 bytes.  A block
// holds the K rows {k, k + 4} (256 elements a row), {k, k + 4, k + 32, k + 36} (128) or {k, k + 4, k + 16, k + 20} and those 32
// further on (64), and the blocks run over k = 0..3, 8..11, 16..19, ... (64: to 11): a ds_read_b64_tr_b16 takes the rows k..k+3 of four blocks for each of its groups of 16 lanes, 32
// bytes of each; the pitch puts eight blocks in a row on different banks, and every fragment of a stage is one register
// plus an immediate away.
#pragma once
#include "gemm_mfma_pipe.hpp"
#include "mfma_wait_counts.hpp"

namespace zluda_amd {

// The lane number, computed where it is used.  Nothing an epilogue needs per lane may stay live across the K loop of a
// 256 x 256 tile: the loop has no register to spare, what is kept is spilled to scratch memory, and a reload from there (like
// every load from memory) first waits for the stages in flight, which are older.
__device__ __forceinline__ int lane_here() {
  int l = 0;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
#endif
  return l;
}

typedef unsigned v2u __attribute__((ext_vector_type(2)));

// ---- epilogues for the 16x16 accumulator layout ------------------------------------------------------
// acc[a][b] is the 16 x 16 tile at (P tile a, Q tile b) of the wave tile; lane l holds elements
// P = 16a + 4*(l/16) + v (v = 0..3), Q = 16b + l%16.

// A lane's store of four consecutive elements along P: where the four end past P's last index it is dropped, and those of
// them that exist are stored one by one.  `left`: P indices from the lane's first one to the end.
__device__ __forceinline__ int store4_offset(int left, int voff) { return left >= 4 ? voff : kStoreNowhere; }
__device__ __forceinline__ int store1_offset(int left, int e, int voff, int esz) { return left < 4 && e < left ? voff + e * esz : kStoreNowhere; }

// raw accumulators (int32 or fp32 bits) of a whole wave tile into a matrix of `pitch` dwords per Q column
// through the window `rs` that starts at the wave tile's corner; EDGE: the tile may hang over the end of P, `p_left` indices
// from the corner
template <bool EDGE, int TP, int TQ, class AccV>
__device__ __forceinline__ void mfma16_store_raw(__amdgpu_buffer_rsrc_t rs, int pitch, AccV (&acc)[TP][TQ], int mul, int p_left) {
  const int lane = lane_here();
  const int voff = ((lane & 15) * pitch + 4 * (lane >> 4)) * 4;
  const bool ragged = EDGE && p_left < TP * 16 && (p_left & 3);  // (uniform) some lane's four straddle the end
#pragma unroll
  for (int b = 0; b < TQ; b++)
#pragma unroll
    for (int a = 0; a < TP; a++) {
      v4i v;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = to_bits(acc[a][b][e]);
      if (mul != 1) v *= mul;
      const int left = p_left - (a * 16 + 4 * (lane >> 4));
      buffer_store_b128_guarded(v, rs, EDGE ? store4_offset(left, voff) : voff, (b * 16 * pitch + a * 16) * 4);
      if (ragged) {
#pragma unroll
        for (int e = 0; e < 3; e++) __builtin_amdgcn_raw_buffer_store_b32(v[e], rs, store1_offset(left, e, voff, 4), (b * 16 * pitch + a * 16) * 4, 0);
      }
    }
}

// float epilogue without a C read: D bf16, f16 or f32 in 16-byte stores, at any element's address and any
// pitch (the memory system takes such stores unaligned).  A tile that hangs over the end of P (EDGE) drops the lanes past it
// and stores the elements of a lane's 16 bytes that straddle the end one by one.
// DT: 0 bf16, 1 f16, 2 f32, -1 one of the 16-bit types; ACT: the activation, -1 any.  Whole tiles have both fixed at compile
// time (int8 4096 x 4096 x 1024 -> bf16 + GELU: 31.3 us with run-time branches per 16 x 16 tile, 28.7).  Edge tiles branch: the
// 64 tiles of a wave are unrolled, and a grid has few of them.
// (us, 8-byte stores and a branch per factor and element before: bf16 4096 x 4096 x 512 27.0 -> 22.4, with a D pitch of 4100 34.6 -> 23.6;
// 32000 x 512 x 1024 with pitches of 32004 49.7 -> 40.8 and 32003 53.2 -> 46.2: stores at 2-byte alignment cost more.)
template <int KIND, int WP, int WQ, int TP, int TQ, int DT, int ACT, bool EDGE, class AccV>
__device__ __forceinline__ void mfma16_store_f(const MfmaParams &prm, AccV (&acc)[TP][TQ], int p0, int q0, int NP, int NQ, int bt, int wave) {
  constexpr int WTP = TP * 16, WTQ = TQ * 16;
  constexpr bool WIDE = DT == 2;
  constexpr int ESZ = WIDE ? 4 : 2;
  const GemmArgs &g = prm.g;
  const int lane = lane_here();
  const int wp = wave % WP, wq = wave / WP;
  Epilogue ep(g, bt);
  const bool swp = prm.swapped != 0;
  const int act = ACT >= 0 ? ACT : (int)g.act;
  const bool to_bf16 = DT >= 0 ? DT == 0 : g.d_type == CUDA_R_16BF;
  const bool ragged = EDGE && NP < p0 + wp * WTP + WTP && (NP & 3);  // (uniform) some lane's four straddle the end of P
  const int d_sq = (int)(swp ? g.d_si : g.d_sj);  // < kNarrowPitch (checked by the dispatcher)
  const int pc = p0 + wp * WTP, qc = q0 + wq * WTQ;
  const int p_left = NP - pc;  // P indices from the wave tile's corner to the end
  const int64_t corner = (int64_t)qc * d_sq + pc;
  char *Dw = (char *)g.D + (g.d_sb * bt + corner) * ESZ;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dw, 0, tile_window_bytes(d_sq, NP, NQ, corner, ESZ), 0x00020000);
  const int voff = ((lane & 15) * d_sq + 4 * (lane >> 4)) * ESZ;
  // The factors along Q (one index per lane and tile column; columns past the end are dropped by the window) and along P (a
  // lane's four consecutive indices of each tile).  Whether a factor is a vector is decided once for all of them: decided
  // where each is used, the kernel is a chain of hundreds of branches around single loads.
  float qs[TQ], qb[TQ], ps[TP][4];
  const float *q_v = swp ? ep.alpha_v : ep.sb_v, *p_v = swp ? ep.sb_v : ep.alpha_v;
  const float q_s = swp ? ep.alpha_s : ep.sb_s, p_s = swp ? ep.sb_s : ep.alpha_s;
  const int q_lane = qc + (lane & 15), p_lane = pc + 4 * (lane >> 4);
#pragma unroll
  for (int b = 0; b < TQ; b++) { qs[b] = q_s; qb[b] = 0.0f; }
#pragma unroll
  for (int a = 0; a < TP; a++)
#pragma unroll
    for (int e = 0; e < 4; e++) ps[a][e] = p_s;
  if (q_v) {
#pragma unroll
    for (int b = 0; b < TQ; b++) qs[b] = q_v[min(q_lane + b * 16, NQ - 1)];
  }
  if (p_v) {
#pragma unroll
    for (int a = 0; a < TP; a++)
#pragma unroll
      for (int e = 0; e < 4; e++) ps[a][e] = p_v[EDGE ? min(p_lane + a * 16 + e, NP - 1) : p_lane + a * 16 + e];
  }
  if (ep.sa_v) {
    if (swp) {
#pragma unroll
      for (int b = 0; b < TQ; b++) qs[b] *= ep.sa_v[min(q_lane + b * 16, NQ - 1)];
    } else {
#pragma unroll
      for (int a = 0; a < TP; a++)
#pragma unroll
        for (int e = 0; e < 4; e++) ps[a][e] *= ep.sa_v[EDGE ? min(p_lane + a * 16 + e, NP - 1) : p_lane + a * 16 + e];
    }
  } else if (swp) {
#pragma unroll
    for (int b = 0; b < TQ; b++) qs[b] *= ep.sa_s;
  } else {
#pragma unroll
    for (int a = 0; a < TP; a++)
#pragma unroll
      for (int e = 0; e < 4; e++) ps[a][e] *= ep.sa_s;
  }
  if (swp && g.bias) {
    uint32_t raw[TQ];
#pragma unroll
    for (int b = 0; b < TQ; b++) raw[b] = ep.bias_raw(min(q_lane + b * 16, NQ - 1));
#pragma unroll
    for (int b = 0; b < TQ; b++) qb[b] = ep.bias_from_raw(raw[b]);
  }
  // the bias, along P (a row-major D: along Q): raw bits of all tiles in one burst, then their values
  float pb[TP][4];
#pragma unroll
  for (int a = 0; a < TP; a++)
#pragma unroll
    for (int e = 0; e < 4; e++) pb[a][e] = 0.0f;
  if (g.bias && !swp) {
    uint32_t raw[TP][4];
    if (g.bias_type == CUDA_R_32F) {
      const uint32_t *v = (const uint32_t *)g.bias + g.bias_sb * bt;
#pragma unroll
      for (int a = 0; a < TP; a++)
#pragma unroll
        for (int e = 0; e < 4; e++) pb[a][e] = bits2f(v[EDGE ? min(p_lane + a * 16 + e, NP - 1) : p_lane + a * 16 + e]);
    } else {
      const uint16_t *v = (const uint16_t *)g.bias + g.bias_sb * bt;
      if (!EDGE && (((uintptr_t)v) & 7) == 0) {  // (rows start at multiples of 4)
        v2i t[TP];
#pragma unroll
        for (int a = 0; a < TP; a++) t[a] = *(const v2i *)(v + p_lane + a * 16);
#pragma unroll
        for (int a = 0; a < TP; a++) {
          raw[a][0] = (uint32_t)t[a][0] & 0xffffu; raw[a][1] = (uint32_t)t[a][0] >> 16;
          raw[a][2] = (uint32_t)t[a][1] & 0xffffu; raw[a][3] = (uint32_t)t[a][1] >> 16;
        }
      } else {
#pragma unroll
        for (int a = 0; a < TP; a++)
#pragma unroll
          for (int e = 0; e < 4; e++) raw[a][e] = v[EDGE ? min(p_lane + a * 16 + e, NP - 1) : p_lane + a * 16 + e];
      }
      if (g.bias_type == CUDA_R_16BF) {
#pragma unroll
        for (int a = 0; a < TP; a++)
#pragma unroll
          for (int e = 0; e < 4; e++) pb[a][e] = dec_bf16((uint16_t)raw[a][e]);
      } else {
#pragma unroll
        for (int a = 0; a < TP; a++)
#pragma unroll
          for (int e = 0; e < 4; e++) pb[a][e] = dec_f16((uint16_t)raw[a][e]);
      }
    }
  }
  // Two tiles along P at a time: the 16-bit results of a lane's four rows are 8 bytes of either, and the lane groups g and g ^ 1
  // trade halves (v_permlane16_swap), after which a lane of an even group holds rows 4g .. 4g + 7 of the first tile and a lane
  // of an odd one rows 4(g-1) .. 4(g-1) + 7 of the second: 16 bytes a lane, 64 contiguous bytes of each of 16 columns.
  static_assert(TP % 2 == 0, "tiles along P are stored in pairs");
  const int grp = lane >> 4, first = (grp & 1) ? 4 * grp + 12 : 4 * grp;  // the lane's first P index inside a pair
  const int voff_pair = ((lane & 15) * d_sq + first) * 2;
#pragma unroll
  for (int a = 0; a < TP; a += 2) {
#pragma unroll
    for (int b = 0; b < TQ; b++) {
      float x[2][4];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float accf = KIND == KIND_I8 ? (float)to_bits(acc[a + h][b][e]) : bits2f((uint32_t)to_bits(acc[a + h][b][e]));
          x[h][e] = ps[a + h][e] * qs[b] * accf + (swp ? qb[b] : pb[a + h][e]);
        }
      if (act == ACT_GELU) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int e = 0; e < 4; e++) x[h][e] = gelu_tanh(x[h][e]);
      } else if (act == ACT_RELU) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int e = 0; e < 4; e++) x[h][e] = x[h][e] > 0.0f ? x[h][e] : 0.0f;
      }
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) x[h][e] *= ep.sd;
      const int soff = (b * 16 * d_sq + a * 16) * ESZ;  // uniform
      if constexpr (WIDE) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int left = NP - (pc + (a + h) * 16 + 4 * (lane >> 4));
          const v4i pk = {(int)f2bits(x[h][0]), (int)f2bits(x[h][1]), (int)f2bits(x[h][2]), (int)f2bits(x[h][3])};
          buffer_store_b128_guarded(pk, rs, EDGE ? store4_offset(left, voff) : voff, soff + h * 16 * ESZ);
          if (ragged) {
#pragma unroll
            for (int e = 0; e < 3; e++) __builtin_amdgcn_raw_buffer_store_b32(pk[e], rs, store1_offset(left, e, voff, 4), soff + h * 16 * ESZ, 0);
          }
        }
      } else {
        uint32_t lo[2], hi[2];  // the first and the second tile
        if (to_bf16) {
          lo[0] = pack_bf16x2(x[0][0], x[0][1]); lo[1] = pack_bf16x2(x[0][2], x[0][3]);
          hi[0] = pack_bf16x2(x[1][0], x[1][1]); hi[1] = pack_bf16x2(x[1][2], x[1][3]);
        } else {
          lo[0] = pack_f16x2(x[0][0], x[0][1]); lo[1] = pack_f16x2(x[0][2], x[0][3]);
          hi[0] = pack_f16x2(x[1][0], x[1][1]); hi[1] = pack_f16x2(x[1][2], x[1][3]);
        }
        v4i pk = {(int)lo[0], (int)lo[1], (int)hi[0], (int)hi[1]};
#if defined(__HIP_DEVICE_COMPILE__)
        const v2u s0 = __builtin_amdgcn_permlane16_swap(lo[0], hi[0], false, false);
        const v2u s1 = __builtin_amdgcn_permlane16_swap(lo[1], hi[1], false, false);
        pk = v4i{(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]};
#endif
        if constexpr (!EDGE) {
          buffer_store_b128_guarded(pk, rs, voff_pair, soff);
        } else {
          const int left = NP - (pc + a * 16 + first);
          buffer_store_b128_guarded(pk, rs, left >= 8 ? voff_pair : kStoreNowhere, soff);
          if (p_left > a * 16 && p_left < a * 16 + 32 && (p_left & 7)) {  // (uniform) some lane's eight straddle the end
#pragma unroll
            for (int e = 0; e < 7; e++)
              __builtin_amdgcn_raw_buffer_store_b16((short)(pk[e >> 1] >> (16 * (e & 1))), rs, left < 8 && e < left ? voff_pair + e * 2 : kStoreNowhere, soff, 0);
          }
        }
      }
    }
  }
}

// the largest divisor of `tq` that does not exceed `fit`
constexpr int staging_columns(int fit, int tq) {
  int c = fit < tq ? fit : tq;
  while (c > 1 && tq % c != 0) c--;
  return c;
}

// everything else (C reads, 8-bit outputs, integer outputs of a float epilogue, integer alpha vectors):
// element by element through the scalar epilogue.  Correct for whatever the planner admits; not fast.
// The accumulators are staged in the wave's share of the (now free) LDS, as many tile columns per pass as
// fit, so that the scalar epilogue is a rolled loop (a function call would do as well, but a call anywhere
// in the kernel makes the compiler keep the kernel arguments in private memory).
// The caller guarantees that every wave of the workgroup is done with the LDS tiles (a barrier behind the
// K loop); `lds_words` / `lds_bytes`: the workgroup's LDS.
template <int KIND, int WP, int WQ, int TP, int TQ, int LDS_BYTES, class AccV>
__device__ __forceinline__ void mfma16_store_general(const MfmaParams &prm, AccV (&acc)[TP][TQ], int *lds_words, int p0, int q0,
                                                     int NP, int NQ, int bt, int wave) {
  constexpr int WTP = TP * 16, WTQ = TQ * 16;
  constexpr int PER_WAVE = LDS_BYTES / (WP * WQ);            // bytes of staging per wave
  constexpr int COLS = staging_columns(PER_WAVE / (16 * WTP * 4), TQ);  // tile columns per pass
  static_assert(COLS >= 1 && TQ % COLS == 0, "staging passes");
  const GemmArgs &g = prm.g;
  const int lane = lane_here();
  const int wp = wave % WP, wq = wave / WP;
  int *stage = lds_words + wave * (PER_WAVE / 4);
  Epilogue ep(g, bt);
  const bool swp = prm.swapped != 0;
#pragma unroll
  for (int pass = 0; pass < TQ / COLS; pass++) {
#pragma unroll
    for (int bb = 0; bb < COLS; bb++)
#pragma unroll
      for (int a = 0; a < TP; a++) {
        v4i v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = to_bits(acc[a][pass * COLS + bb][e]);
        *(v4i *)&stage[(bb * 16 + (lane & 15)) * WTP + a * 16 + 4 * (lane >> 4)] = v;
      }
    // (LDS executes the writes and reads of one wave in program order: no barrier for wave-private rows)
#pragma unroll 1
    for (int e = lane; e < COLS * 16 * WTP; e += 64) {
      const int ql = e / WTP, pl = e % WTP;
      const int pi = p0 + wp * WTP + pl, qi = q0 + wq * WTQ + pass * COLS * 16 + ql;
      if (pi >= NP || qi >= NQ) continue;
      const int raw = stage[ql * WTP + pl];
      const int i = swp ? qi : pi, j = swp ? pi : qi;
      if (g.int_scale) ep.store_int(i, j, raw);
      else ep.store_f(i, j, KIND == KIND_I8 ? (float)raw : bits2f((uint32_t)raw));
    }
  }
}

// GELU with its input kept and GELU's gradient (mfma_store_tile_aux()) in the 16x16 layout: tiles in pairs, the float values trade halves
// as the 16-bit ones do in mfma16_store_f(), after which a lane has eight consecutive P indices: 16 bytes of D and of aux.
template <int WP, int WQ, int TP, int TQ, int MODE, class AccV>
__device__ __forceinline__ void mfma16_store_aux(const MfmaParams &prm, AccV (&acc)[TP][TQ], int p0, int q0, int NP, int NQ, int bt, int wave) {
  constexpr int WTP = TP * 16, WTQ = TQ * 16, PAIRS = TP / 2;
  const GemmArgs &g = prm.g;
  const int lane = lane_here();
  const int wp = wave % WP, wq = wave / WP;
  const int pc = p0 + wp * WTP, qc = q0 + wq * WTQ;
  const EpilogueScalars sc(g);
  const AuxTile at(prm, sc, pc, qc, NP, NQ, bt, q0 / WTQ + wq, prm.tiles_q * WQ);
  const bool bf16 = g.d_type == CUDA_R_16BF;
  const int grp = lane >> 4, first = (grp & 1) ? 4 * grp + 12 : 4 * grp;  // the lane's first P index inside a pair
  const int vd_in = ((lane & 15) * at.d_sq + first) * 2, vx_in = ((lane & 15) * at.x_sq + first) * 2;
  const char *bias = MODE == 1 && g.bias ? (const char *)g.bias + g.bias_sb * bt * (g.bias_type == CUDA_R_32F ? 4 : 2) : nullptr;
  // the bias of a pair's eight rows (1), or their sums (2)
  float row[PAIRS][8];
#pragma unroll
  for (int a = 0; a < PAIRS; a++) {
    const int at_p = min(pc + a * 32 + first, NP - 8);  // the lane's eight P indices exist or do not (their number is a multiple of 8)
#pragma unroll
    for (int e = 0; e < 8; e++) row[a][e] = 0.0f;
    if (MODE == 1 && bias) {
      if (g.bias_type == CUDA_R_32F) {
#pragma unroll
        for (int e = 0; e < 8; e++) row[a][e] = ((const float *)bias)[at_p + e];
      } else {
        uint32_t raw[4];
        if (((uintptr_t)bias & 15) == 0) {
          const v4i t = *(const v4i *)(bias + at_p * 2);
#pragma unroll
          for (int d = 0; d < 4; d++) raw[d] = (uint32_t)t[d];
        } else {
#pragma unroll
          for (int d = 0; d < 4; d++) raw[d] = ((const uint16_t *)bias)[at_p + 2 * d] | (uint32_t)((const uint16_t *)bias)[at_p + 2 * d + 1] << 16;
        }
        const bool bias_bf16 = g.bias_type == CUDA_R_16BF;
#pragma unroll
        for (int d = 0; d < 4; d++) { row[a][2 * d] = low_half(raw[d], bias_bf16); row[a][2 * d + 1] = high_half(raw[d], bias_bf16); }
      }
    }
  }
  // Along P first: a pair of tiles stores 64 bytes of a column, half a line, and with another column's halves in between both matrices' lines left the
  // L2 of an XCD (whose 32 tiles of 256 x 256 are 8 MiB of them) half written: bf16 1480 x 29920 x 176, two batches, GELU_AUX_BIAS 209 us, now 137.
#pragma unroll
  for (int b = 0; b < TQ; b++) {
    // (the column's aux pieces in one burst)
    v4i x_in[PAIRS];
    if constexpr (MODE == 2) {
#pragma unroll
      for (int a = 0; a < PAIRS; a++)
        x_in[a] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(at.rs_x, pc + a * 32 + first < NP ? vx_in : kStoreNowhere, (b * 16 * at.x_sq + a * 32) * 2, 0));
    }
#pragma unroll
    for (int a = 0; a < PAIRS; a++) {
      const bool in = pc + a * 32 + first < NP;
      const int vd = in ? vd_in : kStoreNowhere, vx = in ? vx_in : kStoreNowhere;
      float y[8];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t lo = f2bits(at.factor * bits2f((uint32_t)to_bits(acc[2 * a][b][e]))), hi = f2bits(at.factor * bits2f((uint32_t)to_bits(acc[2 * a + 1][b][e])));
#if defined(__HIP_DEVICE_COMPILE__)
        const v2u s = __builtin_amdgcn_permlane16_swap(lo, hi, false, false);
        y[e] = bits2f(s[0]); y[4 + e] = bits2f(s[1]);
#else
        y[e] = bits2f(lo); y[4 + e] = bits2f(hi);
#endif
      }
      if constexpr (MODE == 1) {
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] += row[a][e];
        v4i keep;
#pragma unroll
        for (int d = 0; d < 4; d++) keep[d] = (int)pack_halves(y[2 * d], y[2 * d + 1], bf16);
        buffer_store_b128_guarded(keep, at.rs_x, vx, (b * 16 * at.x_sq + a * 32) * 2);
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] = gelu_tanh(y[e]) * sc.sd;
      } else {
#pragma unroll
        for (int d = 0; d < 4; d++) {
          y[2 * d] *= dgelu_tanh(low_half((uint32_t)x_in[a][d], bf16));
          y[2 * d + 1] *= dgelu_tanh(high_half((uint32_t)x_in[a][d], bf16));
        }
        // (columns past the end hold products of some column)
        const bool counts = qc + b * 16 + (lane & 15) < NQ;
#pragma unroll
        for (int e = 0; e < 8; e++) row[a][e] += counts ? y[e] : 0.0f;
      }
      v4i pk;
#pragma unroll
      for (int d = 0; d < 4; d++) pk[d] = (int)pack_halves(y[2 * d], y[2 * d + 1], bf16);
      buffer_store_b128_guarded(pk, at.rs_d, vd, (b * 16 * at.d_sq + a * 32) * 2);
      __builtin_amdgcn_sched_barrier(0);  // one pair at a time: what the scheduler hoists across them spills
    }
  }
  if (MODE == 2 && at.sums) {  // over the 16 columns of a lane group
#pragma unroll
    for (int a = 0; a < PAIRS; a++) {
      const int p = pc + a * 32 + first;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        float &t = row[a][e];
        t += bits2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2bits(t), 0x128 /* row_ror:8 */, 0xF, 0xF, true));
        t += bits2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2bits(t), 0x124, 0xF, 0xF, true));
        t += bits2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2bits(t), 0x122, 0xF, 0xF, true));
        t += bits2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2bits(t), 0x121, 0xF, 0xF, true));
      }
      if ((lane & 15) == 0 && p < NP) {
#pragma unroll
        for (int e = 0; e < 8; e++) at.sums[p + e] = row[a][e];
      }
    }
  }
}

// The epilogues that store straight from the accumulators; false: this problem needs the general one
template <int KIND, int WP, int WQ, int TP, int TQ, class AccV>
__device__ __forceinline__ bool mfma16_store_direct(const MfmaParams &prm, AccV (&acc)[TP][TQ], int p0, int q0, int NP, int NQ, int bt, int wave) {
  constexpr int WTP = TP * 16, WTQ = TQ * 16;
  const GemmArgs &g = prm.g;
  const bool swp = prm.swapped != 0;
  const int64_t d_sq = swp ? g.d_si : g.d_sj;
  const bool narrow = d_sq < kNarrowPitch;  // the lane offsets fit 32 bits
  const bool whole = p0 + WP * WTP <= NP;
  if constexpr (KIND == KIND_I8) {
    if (g.int_scale && narrow && g.alpha_mode != VECTOR_DEV && g.beta_mode == SCALAR_VALUE && g.beta_val.i == 0) {
      const int ialpha = g.alpha_mode == SCALAR_VALUE ? g.alpha_val.i : *(const int32_t *)g.alpha_ptr;
      const int pc = p0 + (wave % WP) * WTP, qc = q0 + (wave / WP) * WTQ;
      const int64_t corner = (int64_t)qc * d_sq + pc;
      int32_t *Dw = (int32_t *)g.D + g.d_sb * bt + corner;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dw, 0, tile_window_bytes(d_sq, NP, NQ, corner, 4), 0x00020000);
      if (whole) mfma16_store_raw<false>(rs, (int)d_sq, acc, ialpha, 0);
      else mfma16_store_raw<true>(rs, (int)d_sq, acc, ialpha, NP - pc);
      return true;
    }
  }
  const MfmaParams &late = args_again(prm);
  if (!g.int_scale && narrow && g.beta_mode == SCALAR_VALUE && g.beta_val.f == 0.0f &&
      (g.d_type == CUDA_R_16BF || g.d_type == CUDA_R_16F || g.d_type == CUDA_R_32F)) {
#define ZLUDA_EPI16(DT_, ACT_, EDGE_) mfma16_store_f<KIND, WP, WQ, TP, TQ, DT_, ACT_, EDGE_>(late, acc, p0, q0, NP, NQ, bt, wave)
#define ZLUDA_EPI16_ACT(DT_)                                 \
  if (g.act == ACT_GELU) ZLUDA_EPI16(DT_, ACT_GELU, false);  \
  else if (g.act == ACT_RELU) ZLUDA_EPI16(DT_, ACT_RELU, false); \
  else ZLUDA_EPI16(DT_, ACT_NONE, false);
    if (!whole) {
      if (g.d_type == CUDA_R_32F) ZLUDA_EPI16(2, -1, true);
      else ZLUDA_EPI16(-1, -1, true);
    } else if (g.d_type == CUDA_R_16BF) {
      ZLUDA_EPI16_ACT(0)
    } else if (g.d_type == CUDA_R_16F) {
      ZLUDA_EPI16_ACT(1)
    } else {
      ZLUDA_EPI16_ACT(2)
    }
#undef ZLUDA_EPI16_ACT
#undef ZLUDA_EPI16
    return true;
  }
  return false;
}

// AUX: as in mfma_store_tile()
template <int KIND, int WP, int WQ, int TP, int TQ, int LDS_BYTES, bool AUX, class AccV>
__device__ __forceinline__ void mfma16_store_tile(const MfmaParams &prm, AccV (&acc)[TP][TQ], int *lds_words, int p0, int q0, int NP,
                                                  int NQ, int bt, int wave) {
  if constexpr (AUX) {
    static_assert(kind_is_h16(KIND), "aux_in_epilogue()");
    const MfmaParams &late = args_again(prm);
    if (prm.g.act == ACT_GELU_KEPT) mfma16_store_aux<WP, WQ, TP, TQ, 1>(late, acc, p0, q0, NP, NQ, bt, wave);
    else mfma16_store_aux<WP, WQ, TP, TQ, 2>(late, acc, p0, q0, NP, NQ, bt, wave);
    return;
  }
  if (mfma16_store_direct<KIND, WP, WQ, TP, TQ>(prm, acc, p0, q0, NP, NQ, bt, wave)) return;
  __syncthreads();  // (workgroup-uniform branch) the LDS tiles become staging
  mfma16_store_general<KIND, WP, WQ, TP, TQ, LDS_BYTES>(args_again(prm), acc, lds_words, p0, q0, NP, NQ, bt, wave);
}

// ---- the kernel ----------------------------------------------------------------------------------------
// An MC operand's block of LDS (head of this file): the K row of its first lane, and where K row `k` & 36 lies in its block
__host__ __device__ constexpr int mc_block_k(int blk) { return (blk & 3) + 8 * ((blk >> 2) & 3) + 32 * (blk >> 4); }
constexpr int kMcPitch = 1056;
// the K row of a lane's 16 bytes in a block of operands of `rows` rows, less its first lane's
__host__ __device__ constexpr int mc_lane_k(int rows, int lane) {
  return rows == 256 ? 4 * (lane >> 5) : rows == 128 ? 4 * ((lane >> 4) & 1) + 32 * (lane >> 5) : 4 * ((lane >> 3) & 1) + 16 * ((lane >> 4) & 1) + 32 * (lane >> 5);
}
// where the lane group g4 finds the K rows 8 g4 .. 8 g4 + 3 of a stage: row r of them in bytes
__host__ __device__ constexpr int mc_frag_at(int rows, int g4, int r) {
  return rows == 64 ? (r + 4 * (g4 & 1)) * kMcPitch + (g4 >> 1) * 256 : (r + 4 * g4) * kMcPitch;
}
// The chunk swizzle of a K-contiguous operand beside an MC one, whose lane groups hold the K bytes 16 g and 64 + 16 g of a stage: the
// neighbouring chunks of two lane groups fall on different banks with this one
__device__ __forceinline__ int swz_mixed(int r) { return r & 6; }
typedef short v4s_tr __attribute__((ext_vector_type(4)));

// four K elements of one row of an MC operand: 16 lanes, each with the address of 8 bytes (lane 4r + c: K row r, elements
// 4c .. 4c+3), get the K rows 0..3 of element `lane`
__device__ __forceinline__ v2i lds_read_tr16(const char *src) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s_tr *)src));
#else
  return v2i{0, 0};
#endif
}

// lds_dma16() where ds_read_b64_tr_b16 reads what it brings: the compiler would put s_waitcnt vmcnt(0) in front of every
// such read that follows the builtin (it does not follow which slot is read), i.e. wait for the stage just requested.  The
// waits for it are the kernel's own.  The wait states: after M0, and for a resource or offset that came out of a VALU
// instruction (v_readlane of a spilled SGPR).
__device__ __forceinline__ void lds_dma16_uncounted(v4i rs, const void *lds_dst, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t dst = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)lds_dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(dst), "v"(voff), "s"(rs), "s"(soff) : "m0");
#endif
}

template <int KIND, int FQ, int FP, int BP, int BQ, int WP, int WQ, bool PMC = false, bool QMC = false, int NSTAGE = 2, bool AUX = false>
__global__ __launch_bounds__(WP *WQ * 64) void gemm_mfma_pipe16_kernel(MfmaParams prm) {
  static_assert(!(PMC || QMC) || kind_is_h16(KIND), "the transposing LDS reads are those of 16-bit elements");
  static_assert((!PMC || BP == 256 || BP == 128 || BP == 64) && (!QMC || BQ == 256 || BQ == 128 || BQ == 64), "rows of 1 KiB / 2, / 4 or / 8");
  static_assert(KIND == KIND_I8 || KIND == KIND_F8 || kind_is_h16(KIND), "int8, fp8, f16 and bf16 operands");
  constexpr int ESZ = kind_esz(KIND);          // f16 / bf16: the byte geometry of int8 (v_mfma_f32_16x16x32_*: 16 bytes of K per lane)
  constexpr int NT = WP * WQ * 64, NWV = NT / 64;
  constexpr int BKB = 128, CPR = 8, RPW = 8;
  constexpr Pipe16Counts PC = pipe16_counts(BP, BQ, WP, WQ, NSTAGE);  // (shared with the host program that checks the waits)
  constexpr int RPP = PC.rpp;                  // rows filled per DMA pass of the workgroup
  constexpr int LP = PC.lp, LQ = PC.lq;        // DMA instructions per thread, stage and operand
  constexpr int NLOAD = PC.nload;
  static_assert(RPP == NWV * RPW, "eight rows per DMA instruction");
  constexpr int WTP = BP / WP, WTQ = BQ / WQ, TP = WTP / 16, TQ = WTQ / 16;
  constexpr int HP = TP / 2, HQ = TQ / 2;      // fragments per half of the wave tile
  constexpr int KS = KIND == KIND_F8 ? 1 : 2;  // MFMAs per fragment pair (K halves of the 128-byte stage)
  // one slot in 16-byte words: P rows, then Q rows
  constexpr int P_V4 = PMC ? BP / 8 * (kMcPitch / 16) : BP * CPR, Q_V4 = QMC ? BQ / 8 * (kMcPitch / 16) : BQ * CPR;
  constexpr int STAGE_V4 = P_V4 + Q_V4;
  static_assert(BP % RPP == 0 && BQ % RPP == 0, "tile / copy-pass mismatch");
  static_assert(WTP % 32 == 0 && WTQ % 32 == 0, "wave tiles start on multiples of 32 rows (fragment swizzle)");
  static_assert(NSTAGE * STAGE_V4 * 16 <= 160 * 1024, "LDS capacity");
  using acc_v = typename std::conditional<KIND == KIND_I8, v4i, v4f>::type;
  using frag_v = typename std::conditional<KIND != KIND_F8, v4i, v8i>::type;
  struct Frag { frag_v k[KS]; };

  __shared__ v4i lds[NSTAGE * STAGE_V4];

  fetch_args(prm);
  const GemmArgs &g = prm.g;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wp = wave % WP, wq = wave / WP;
  const int r16 = lane & 15, g4 = lane >> 4;

  const WorkItem item = work_item(prm);
  const int bt = item.bt;
  const int p0 = item.p * BP, q0 = item.q * BQ;

  const int NP = prm.swapped ? g.N : g.M, NQ = prm.swapped ? g.M : g.N;
  const int Kbytes = g.K * ESZ;
  const uint8_t *Pg, *Qg;
  int ldp, ldq;
  if (!prm.swapped) {
    Pg = (const uint8_t *)g.A + g.a_sb * bt * ESZ; ldp = (int)(PMC ? g.a_sk : g.a_si) * ESZ;
    Qg = (const uint8_t *)g.B + g.b_sb * bt * ESZ; ldq = (int)(QMC ? g.b_sk : g.b_sj) * ESZ;
  } else {
    Pg = (const uint8_t *)g.B + g.b_sb * bt * ESZ; ldp = (int)(PMC ? g.b_sk : g.b_sj) * ESZ;
    Qg = (const uint8_t *)g.A + g.a_sb * bt * ESZ; ldq = (int)(QMC ? g.a_sk : g.a_si) * ESZ;
  }
  // split-K: this workgroup's share of the stages starts k0 bytes into every row
  int Kbytes_local = Kbytes, k0 = 0;
  if (!AUX && prm.splits > 1) {
    k0 = item.z * prm.split_stages * BKB;
    Kbytes_local = max(0, min(Kbytes - k0, prm.split_stages * BKB));
  }
  const int KT = (Kbytes_local + BKB - 1) / BKB;  // real stages

  // 2 GiB raw buffer windows: an offset with bit 31 set is out of range and reads as zero (the lanes of a
  // K tail)
  const __amdgpu_buffer_rsrc_t rsP = __builtin_amdgcn_make_buffer_rsrc((void *)Pg, 0, 0x80000000, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsQ = __builtin_amdgcn_make_buffer_rsrc((void *)Qg, 0, 0x80000000, 0x00020000);

  // DMA: one wave instruction fills 8 rows x 128 bytes; lane l -> row l / 8, slot l % 8, global chunk
  // slot ^ swizzle(row)
  const int dr = lane / CPR, dslot = lane % CPR;
  const int drow = wave * RPW + dr;  // passes advance by RPP, a multiple of 32: same swizzle
  const int dcg = dslot ^ (PMC || QMC ? swz_mixed(drow) : swz(drow));
  int voffP[LP], voffQ[LQ];
  // MC: an instruction fills a block; lane l -> K row and 16-byte piece of it.  A piece past the last one of the row index
  // loads that one (rows past the end of D are dropped), which holds at least one element of the operand: with the
  // 16-byte aligned pitch the planner asks for it lies in the operand's own 16-byte granules.
  const int mkP = mc_block_k(wave) + mc_lane_k(BP, lane), mkQ = mc_block_k(wave) + mc_lane_k(BQ, lane);
#pragma unroll
  for (int i = 0; i < LP; i++)
    if constexpr (PMC) voffP[i] = i ? 0 : mkP * ldp + min(p0 + 8 * (lane & (BP / 8 - 1)), (NP - 1) & ~7) * ESZ;
    else voffP[i] = min(p0 + drow + RPP * i, NP - 1) * ldp + dcg * 16;
#pragma unroll
  for (int i = 0; i < LQ; i++)
    if constexpr (QMC) voffQ[i] = i ? 0 : mkQ * ldq + min(q0 + 8 * (lane & (BQ / 8 - 1)), (NQ - 1) & ~7) * ESZ;
    else voffQ[i] = min(q0 + drow + RPP * i, NQ - 1) * ldq + dcg * 16;
  const int tail_bytes = Kbytes_local - (KT - 1) * BKB;
  const int oob_last = dcg * 16 < tail_bytes ? 0 : (int)0x80000000;

  const v4i rawP = {(int)(uintptr_t)Pg, (int)((uintptr_t)Pg >> 32) & 0xffff, (int)0x80000000, 0x00020000};
  const v4i rawQ = {(int)(uintptr_t)Qg, (int)((uintptr_t)Qg >> 32) & 0xffff, (int)0x80000000, 0x00020000};
  constexpr bool MC = PMC || QMC;

  // stage kt -> LDS slot at 16-byte offset `so`, DMA instruction `n` of LP + LQ.  Stages kt >= KT are never multiplied; they
  // are issued only so that every stage has the same vector memory operations in flight, as real loads of one cache
  // line (an instruction whose lanes are all out of range completes without a memory round trip and can
  // retire ahead of older loads).  Rings of more than two slots drain where such a stage would be in flight, and request none.
  auto issue_one = [&](int kt, int so, auto n_c) {
    constexpr int n = decltype(n_c)::value;
    constexpr bool is_p = n < LP, mc = is_p ? PMC : QMC;
    constexpr int i = is_p ? n : n - LP;
    const int live = NSTAGE > 2 || kt < KT ? -1 : 0;  // uniform
    const int *voff = is_p ? voffP : voffQ;
    v4i *base = &lds[so] + (is_p ? 0 : P_V4);
    if constexpr (mc) {
      // K rows from `klim` on are past the end (an offset of bit 31 alone, which no stage's offset carries beyond 2^32);
      // the blocks of a wave lie whole K rows apart: in the scalar offset
      const int klim = kt == KT - 1 ? tail_bytes / ESZ : BKB / ESZ;
      const int vo = ((is_p ? mkP : mkQ) < klim - mc_block_k(i * NWV) ? voff[0] : (int)0x80000000) & live;
      const int soff = (((k0 + kt * BKB) / ESZ + mc_block_k(i * NWV)) & live) * (is_p ? ldp : ldq);
      lds_dma16_uncounted(is_p ? rawP : rawQ, base + (wave + NWV * i) * (kMcPitch / 16), vo, soff);
    } else {
      const int oob = kt == KT - 1 ? oob_last : 0;
      const int soff = (k0 + kt * BKB) & live;
      v4i *dst = base + (wave * RPW + RPP * i) * CPR;
      if constexpr (MC) lds_dma16_uncounted(is_p ? rawP : rawQ, dst, (voff[i] | oob) & live, soff);
      else lds_dma16(is_p ? rsP : rsQ, dst, (voff[i] | oob) & live, soff);
    }
  };
  auto issue_stage = [&](int kt, int so) { static_for<NLOAD>([&](auto n_c) { issue_one(kt, so, n_c); }); };
  // the same for a stage that neither ends K nor lies behind its end (operands along their row index)
  auto issue_inside = [&](int kt, int so, auto n_c) {
    constexpr int n = decltype(n_c)::value;
    constexpr bool is_p = n < LP, mc = is_p ? PMC : QMC;
    constexpr int i = is_p ? n : n - LP;
    const int *voff = is_p ? voffP : voffQ;
    v4i *base = &lds[so] + (is_p ? 0 : P_V4);
    if constexpr (mc) {
      const int ld = is_p ? ldp : ldq;
      lds_dma16_uncounted(is_p ? rawP : rawQ, base + (wave + NWV * i) * (kMcPitch / 16), voff[0], (k0 + kt * BKB) / ESZ * ld + mc_block_k(i * NWV) * ld);
    } else {
      lds_dma16_uncounted(is_p ? rawP : rawQ, base + (wave * RPW + RPP * i) * CPR, voff[i], k0 + kt * BKB);
    }
  };

  // ---- fragment addressing --------------------------------------------------------------------------------
  // Tiles start on multiples of 16 rows; the swizzle depends on the row mod 32, so even and odd tiles
  // differ.  [tile parity][first / second 16-byte piece of the lane] in 16-byte words inside a slot
  int fragP[2][2], fragQ[2][2];
#pragma unroll
  for (int par = 0; par < 2; par++)
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
      const int row = par * 16 + r16;
      const int ch = PMC || QMC ? (4 * kk + g4) ^ swz_mixed(row) : (2 * g4 + kk) ^ swz(row);
      fragP[par][kk] = (wp * WTP + row) * CPR + ch;
      // (summed in this order: the other one has the compiler hoist two more addresses than the loop has registers for, and
      // their reloads cost 7 % of int8 and bf16 8192 x 4096 x 1024)
      fragQ[par][kk] = PMC ? P_V4 + (wq * WTQ + row) * CPR + ch : (BP + wq * WTQ + row) * CPR + ch;
    }
  // MC: K row 8 * (l / 16) + (l % 16) / 4, elements 4 * (l % 4) .. +3 of the wave tile, in bytes inside a slot
  const int mfragP = mc_frag_at(BP, g4, r16 >> 2) + 8 * (r16 & 3) + wp * WTP * 2;
  const int mfragQ = P_V4 * 16 + mc_frag_at(BQ, g4, r16 >> 2) + 8 * (r16 & 3) + wq * WTQ * 2;
  // 16-row tile `tile` of the wave tile, from the stage in the slot at `so`
  auto load_frag = [&](int so, const int (&fr)[2][2], auto tile_c, Frag &f) {
    constexpr int tile = decltype(tile_c)::value;
    const v4i *base = &lds[so + (tile >> 1) * 32 * CPR];
    const v4i lo = base[fr[tile & 1][0]], hi = base[fr[tile & 1][1]];
    if constexpr (KIND == KIND_F8) {
      f.k[0] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
      f.k[0] = lo;
      f.k[1] = hi;
    }
  };

  auto load_frag_mc = [&](int so, int fr, auto rows_c, auto tile_c, Frag &f) {
    constexpr int B = decltype(rows_c)::value, tile = decltype(tile_c)::value;
    constexpr int UP4 = B * 2, UP32 = B == 256 ? 16 * kMcPitch : 512;  // bytes to the K row 4 / 32 further on
    const char *base = (const char *)&lds[so] + fr + tile * 32;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const v2i lo = lds_read_tr16(base + ks * UP32), hi = lds_read_tr16(base + ks * UP32 + UP4);
      f.k[ks] = frag_v{lo[0], lo[1], hi[0], hi[1]};
    }
  };

  acc_v acc[TP][TQ];
#pragma unroll
  for (int a = 0; a < TP; a++)
#pragma unroll
    for (int b = 0; b < TQ; b++)
#pragma unroll
      for (int v = 0; v < 4; v++) acc[a][b][v] = 0;

  Frag pf[2][HP], qf[2][HQ];  // [half of the wave tile][fragment]
  // fragments [I0, I1) of P half h
  auto load_p_part = [&](int so, auto h_c, auto i0_c, auto i1_c) {
    constexpr int h = decltype(h_c)::value, I0 = decltype(i0_c)::value, I1 = decltype(i1_c)::value;
    static_for<I1 - I0>([&](auto i_c) {
      constexpr int i = I0 + decltype(i_c)::value;
      if constexpr (PMC) load_frag_mc(so, mfragP, std::integral_constant<int, BP>{}, std::integral_constant<int, h * HP + i>{}, pf[h][i]);
      else load_frag(so, fragP, std::integral_constant<int, h * HP + i>{}, pf[h][i]);
    });
  };
  auto load_p_half = [&](int so, auto h_c) {
    load_p_part(so, h_c, std::integral_constant<int, 0>{}, std::integral_constant<int, HP>{});
  };
  auto load_q_half = [&](int so, auto h_c) {
    constexpr int h = decltype(h_c)::value;
    static_for<HQ>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      if constexpr (QMC) load_frag_mc(so, mfragQ, std::integral_constant<int, BQ>{}, std::integral_constant<int, h * HQ + i>{}, qf[h][i]);
      else load_frag(so, fragQ, std::integral_constant<int, h * HQ + i>{}, qf[h][i]);
    });
  };
  // the MFMAs of P half ph against Q half qh; K half by K half, so that the two instructions of a tile
  // (int8) are a whole sub-step's worth of independent instructions apart
  auto mfma_part = [&](auto ph_c, auto qh_c, auto n0_c, auto n1_c) {  // number n0 .. n1 - 1 of them
    constexpr int ph = decltype(ph_c)::value, qh = decltype(qh_c)::value;
#pragma unroll
    for (int n = decltype(n0_c)::value; n < decltype(n1_c)::value; n++) {
          const int ks = n / (HP * HQ), x = n % (HP * HQ), i = x / HQ, j = x % HQ;
          acc_v &c = acc[ph * HP + i][qh * HQ + j];
          if constexpr (KIND == KIND_I8) c = __builtin_amdgcn_mfma_i32_16x16x64_i8(pf[ph][i].k[ks], qf[qh][j].k[ks], c, 0, 0, 0);
          else if constexpr (KIND == KIND_F16)
            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, pf[ph][i].k[ks]), __builtin_bit_cast(v8h, qf[qh][j].k[ks]), c, 0, 0, 0);
          else if constexpr (KIND == KIND_BF16)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, pf[ph][i].k[ks]), __builtin_bit_cast(v8b, qf[qh][j].k[ks]), c, 0, 0, 0);
          else c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(pf[ph][i].k[ks], qf[qh][j].k[ks], c, FP, FQ, 0, 0, 0, 0);
    }
  };
  auto mfma_halves = [&](auto ph_c, auto qh_c) {
    mfma_part(ph_c, qh_c, std::integral_constant<int, 0>{}, std::integral_constant<int, HP * HQ * KS>{});
  };
  // issue order of a sub-step: its NM MFMAs back to back, with the NDS fragment reads slotted PER_DS at a
  // time behind the first ones (what they fetch is needed one sub-step later, or by the barrier) and the
  // NVM DMA instructions behind the MFMAs that follow
  auto pattern = [&](auto nds_c, auto nvm_c) {
    constexpr int NM = HP * HQ * KS, NDS = decltype(nds_c)::value, NVM = decltype(nvm_c)::value;
    constexpr int PER_DS = 2;  // (1 and 4 per MFMA both measured slower)
    constexpr int MD = (NDS + PER_DS - 1) / PER_DS < NM ? (NDS + PER_DS - 1) / PER_DS : NM;  // MFMAs with reads behind them
    constexpr int MV = NM - MD > 0 ? NM - MD : 1;
    static_for<NM>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      if constexpr (i < MD) {
        constexpr int n = NDS * (i + 1) / MD - NDS * i / MD;
        if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x100, n, 0);  // DS reads
      }
      if constexpr (i >= NM - MV && NVM > 0) {
        constexpr int j = i - (NM - MV), n = NVM * (j + 1) / MV - NVM * j / MV;
        if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x010, n, 0);  // VMEM (LDS DMA)
      }
    });
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- prologue: the first NSTAGE stages in flight, stage 0 landed, its first fragments in registers ---------
  static_for<NSTAGE>([&](auto s_c) {
    if (NSTAGE == 2 || decltype(s_c)::value < KT) issue_stage(decltype(s_c)::value, decltype(s_c)::value * STAGE_V4);
  });
  // (MC: an instruction of the last stage's K tail may hold no K row that exists and retires early, so nothing is counted
  // where one is in flight)
  if (pipe16_drains_prologue(MC, KT, NSTAGE)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  wait_vmcnt_barrier<PC.wait_prologue>();
  load_p_half(0, std::integral_constant<int, 0>{});
  load_q_half(0, std::integral_constant<int, 0>{});

  // ---- one stage ----------------------------------------------------------------------------------------------
  // ODD = 0: on entry P half 0 and Q half 0 of the stage are in registers; the next stage will find P half 0
  // and Q half 1 of its own.  ODD = 1: the same with the Q halves exchanged.
  // `requests`: stage kt + NSTAGE, masked (0), as one inside K (1), or nothing (2: none is left, and what is in flight has to land)
  auto do_stage = [&](int kt, int so, int so_next, auto odd_c, auto requests_c) {
    constexpr int REQ = decltype(requests_c)::value;
    constexpr int QA = decltype(odd_c)::value, QB_ = 1 - QA;  // the Q half that is resident / that is fetched
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    using QAc = std::integral_constant<int, QA>;
    using QBc = std::integral_constant<int, QB_>;
    constexpr int PD = PMC ? 4 : 2, QD = QMC ? 4 : 2;  // LDS reads per fragment
    constexpr int DSP = PD * HP, DSQ = QD * HQ;        // and per half
    // The fragment reads are spread over the four sub-steps (the LDS is the busiest unit of the loop: 24 KiB
    // per wave and stage): EARLY fragments of P half 1 come with QB, LATE fragments of the next stage's P
    // half 0 with its first Q half.
    constexpr int EARLY = 1, LATE = 1;  // (0 / 0: 1.5 % slower at 8192^3 int8; 2 / 1: no better; whole halves early: far slower)
    using I0 = std::integral_constant<int, 0>;
    using IE = std::integral_constant<int, EARLY>;
    using IL = std::integral_constant<int, HP - LATE>;
    using IH = std::integral_constant<int, HP>;
    // (P0, QA) while QB arrives
    load_q_half(so, QBc{});
    load_p_part(so, P1{}, I0{}, IE{});
    mfma_halves(P0{}, QAc{});
    pattern(std::integral_constant<int, DSQ + PD * EARLY>{}, std::integral_constant<int, 0>{});
    // (P0, QB) while P1 arrives
    load_p_part(so, P1{}, IE{}, IH{});
    mfma_halves(P0{}, QBc{});
    pattern(std::integral_constant<int, DSP - PD * EARLY>{}, std::integral_constant<int, 0>{});
    // every fragment of the stage has been requested: wait for them and for this wave's share of stage
    // kt+1, meet the other waves; then the slot is free and the other one readable
    if constexpr (REQ == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    wait_vmcnt_barrier<PC.wait_stage>();
    // (P1, QB): refill this slot with stage kt+NSTAGE, P half 0 of stage kt+1 arrives
    load_p_part(so_next, P0{}, I0{}, IL{});
    if constexpr (MC) {
      // (the scheduler does not know the asm for a memory instruction: its place among the MFMAs is written out)
      constexpr int NM = HP * HQ * KS;
      static_for<NLOAD>([&](auto n_c) {
        constexpr int n = decltype(n_c)::value;
        mfma_part(P1{}, QBc{}, std::integral_constant<int, NM * n / NLOAD>{}, std::integral_constant<int, NM * (n + 1) / NLOAD>{});
        if constexpr (REQ == 1) issue_inside(kt + NSTAGE, so, n_c);
        else if constexpr (REQ == 0) issue_one(kt + NSTAGE, so, n_c);
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      issue_stage(kt + NSTAGE, so);
      mfma_halves(P1{}, QBc{});
      pattern(std::integral_constant<int, DSP - PD * LATE>{}, std::integral_constant<int, NLOAD>{});
    }
    // (P1, QA): Q half QB of stage kt+1 arrives (that stage starts with it)
    load_p_part(so_next, P0{}, IL{}, IH{});
    load_q_half(so_next, QBc{});
    mfma_halves(P1{}, QAc{});
    pattern(std::integral_constant<int, DSQ + PD * LATE>{}, std::integral_constant<int, 0>{});
  };

  int kt = 0;
  using E = std::integral_constant<int, 0>;  // an even stage; masked requests
  using O = std::integral_constant<int, 1>;  // an odd one
  if constexpr (NSTAGE == 2) {
    for (; kt + 2 <= KT; kt += 2) {
      do_stage(kt, 0, STAGE_V4, E{}, E{});
      do_stage(kt + 1, STAGE_V4, 0, O{}, E{});
    }
    if (kt < KT) do_stage(kt, 0, STAGE_V4, E{}, E{});
  } else {
    static_assert(MC, "issue_inside()");
    // Whole turns of the ring with its slots fixed at compile time and without the masks of the last stages: with the slot in a register
    // and the masks a stage of a 64 x 64 tile has 42 scalar and 15 vector instructions beside its 8 MFMAs, a lone workgroup's time
    constexpr int TURN = pipe16_turn(NSTAGE);
    auto turn = [&](auto stage) {
      static_for<TURN>([&](auto u_c) {
        constexpr int u = decltype(u_c)::value;
        stage(kt + u, u % NSTAGE * STAGE_V4, (u + 1) % NSTAGE * STAGE_V4, std::integral_constant<int, u & 1>{});
      });
    };
    for (; pipe16_inside(kt, KT, NSTAGE); kt += TURN)
      turn([&](int k, int so, int so_next, auto odd_c) { do_stage(k, so, so_next, odd_c, std::integral_constant<int, 1>{}); });
    for (; kt < KT; kt += TURN)
      turn([&](int k, int so, int so_next, auto odd_c) {
        if (!pipe16_drains_stage(k, KT, NSTAGE)) do_stage(k, so, so_next, odd_c, std::integral_constant<int, 0>{});
        else if (k < KT) do_stage(k, so, so_next, odd_c, std::integral_constant<int, 2>{});
      });
  }

  __builtin_amdgcn_s_waitcnt(0);  // every DMA of the padding stages has landed before the LDS is reused or the wave ends
  if (!AUX && prm.splits > 1) {
    const int ws_np = prm.tiles_p * BP, ws_nq = prm.tiles_q * BQ;
    int32_t *ws_tile = (int32_t *)prm.ws + ((int64_t)item.z * g.batch + bt) * ws_np * ws_nq + (int64_t)(q0 + wq * WTQ) * ws_np + p0 + wp * WTP;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)ws_tile, 0, 0xFFFFFFFF, 0x00020000);
    mfma16_store_raw<false>(rs, ws_np, acc, 1, 0);
    return;
  }
  mfma16_store_tile<KIND, WP, WQ, TP, TQ, (int)sizeof(lds), AUX>(prm, acc, (int *)&lds[0], p0, q0, NP, NQ, bt, wave);
}

} // namespace zluda_amd
