// MFMA GEMM for K-contiguous f16 / bf16 operands of at most 128 elements of K, on gfx950: many tiles of little work each, such
// as the scores of attention (query times key).
//
// Such a problem is bound by its stores of D (bf16 1000 x 1000 x 128, 64 batches: 128 MB of D, 32 MB of operands).  The tile
// kernels with one tile per workgroup spend most of a tile's time on its launch, its arguments and the round trip of its first
// loads; the four-wave kernel (gemm_mfma_w4.hpp) starts a tile only when the stores of the one before it have
// drained.  Here two workgroups per CU walk runs of 128 x 128 tiles, four waves of 64 x 64:
//   * A run goes along Q, so the P operand's 128 rows stay in registers (as fragments) until its end.
//   * Operand panels (128 rows x all of K, NC chunks of 128 bytes each) come through a ring of two LDS slots, in the order in
//     which they are used; a panel's fragments go to registers, then its slot takes the panel after the next one, so that
//     two of them are on their way during the MFMAs and stores of a tile.
//   * The wait for a panel leaves in flight what was requested or stored after it: the next panel, and the stores of the two
//     tiles in between as far as those were whole tiles (a counted wait must not count stores that are dropped, they can
//     retire early: mfma_wait_counts.hpp).
// While one workgroup of a CU stores, the other one multiplies.
// Measured (MI355X, us, before: the tile kernels): bf16 1000 x 1000 x 128, 64 batches 91 -> 51 (its stores alone, from a kernel that does
// nothing else, in this order 31; without them 18); 512 x 512 x 64, 128 batches 50 -> 22; 4096 x 1024 x 128, 16 batches 72 -> 45.
#pragma once
#include "gemm_mfma_pipe16.hpp"

namespace zluda_amd {

// D = acc * scale * sd, D bf16, f16 (DT 0, 1: tiles in pairs, 16 bytes a lane, as mfma16_store_f) or f32 (2); EDGE: the wave tile
// may hang over the end of P
template <int TP, int TQ, int DT, bool EDGE>
__device__ __forceinline__ void short_store(__amdgpu_buffer_rsrc_t rs, int d_sq, v4f (&acc)[TP][TQ], float scale, float sd, int p_left) {
  const int lane = lane_here(), grp = lane >> 4, first = (grp & 1) ? 4 * grp + 12 : 4 * grp;
  const int voff = DT == 2 ? ((lane & 15) * d_sq + 4 * grp) * 4 : ((lane & 15) * d_sq + first) * 2;
#pragma unroll
  for (int a = 0; a < TP; a += 2)
#pragma unroll
    for (int b = 0; b < TQ; b++) {
      float x[2][4];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) x[h][e] = (scale * acc[a + h][b][e] + 0.0f) * sd;  // (no -0: the other epilogues add a bias of zero)
      if constexpr (DT == 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int left = p_left - (a + h) * 16 - 4 * grp, soff = (b * 16 * d_sq + (a + h) * 16) * 4;
          const v4i pk = {(int)f2bits(x[h][0]), (int)f2bits(x[h][1]), (int)f2bits(x[h][2]), (int)f2bits(x[h][3])};
          buffer_store_b128_guarded(pk, rs, EDGE ? store4_offset(left, voff) : voff, soff);
          if (EDGE && p_left > (a + h) * 16 && p_left < (a + h) * 16 + 16 && (p_left & 3)) {  // (uniform)
#pragma unroll
            for (int e = 0; e < 3; e++) __builtin_amdgcn_raw_buffer_store_b32(pk[e], rs, store1_offset(left, e, voff, 4), soff, 0);
          }
        }
      } else {
        uint32_t lo[2], hi[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          lo[i] = DT == 0 ? pack_bf16x2(x[0][2 * i], x[0][2 * i + 1]) : pack_f16x2(x[0][2 * i], x[0][2 * i + 1]);
          hi[i] = DT == 0 ? pack_bf16x2(x[1][2 * i], x[1][2 * i + 1]) : pack_f16x2(x[1][2 * i], x[1][2 * i + 1]);
        }
        v4i pk = {(int)lo[0], (int)lo[1], (int)hi[0], (int)hi[1]};
#if defined(__HIP_DEVICE_COMPILE__)
        const v2u s0 = __builtin_amdgcn_permlane16_swap(lo[0], hi[0], false, false);
        const v2u s1 = __builtin_amdgcn_permlane16_swap(lo[1], hi[1], false, false);
        pk = v4i{(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]};
#endif
        const int left = p_left - a * 16 - first, soff = (b * 16 * d_sq + a * 16) * 2;
        buffer_store_b128_guarded(pk, rs, EDGE && left < 8 ? kStoreNowhere : voff, soff);
        if (EDGE && p_left > a * 16 && p_left < a * 16 + 32 && (p_left & 7)) {  // (uniform) some lane's eight straddle the end
#pragma unroll
          for (int e = 0; e < 7; e++)
            __builtin_amdgcn_raw_buffer_store_b16((short)(pk[e >> 1] >> (16 * (e & 1))), rs, left < 8 && e < left ? voff + e * 2 : kStoreNowhere, soff, 0);
        }
      }
    }
}

template <int KIND, int NC>
__global__ __launch_bounds__(256, 2) void gemm_mfma_short_kernel(MfmaParams prm) {
  constexpr int BP = 128, BQ = 128, WP = 2, WQ = 2, CPR = 8;
  static_assert(kind_is_h16(KIND) && NC >= 1 && NC <= 2, "f16 and bf16, one or two chunks of 64 elements");
  static_assert(BP == BQ, "one panel geometry");
  constexpr int ESZ = 2;
  constexpr int WTP = BP / WP, WTQ = BQ / WQ, TP = WTP / 16, TQ = WTQ / 16;
  constexpr int KS = 2;                             // MFMAs per fragment pair and chunk
  constexpr int CHUNK_V4 = BP * CPR, SLOT_V4 = NC * CHUNK_V4;
  constexpr int LD = BP / 32;                       // DMA instructions per wave and chunk: 8 rows each, 32 per pass of the workgroup
  constexpr ShortCounts SC = short_counts(NC);      // (mfma_wait_counts.hpp, where a host program replays the waits)
  static_assert(SC.panel == NC * LD && SC.stores == TP * TQ / 2, "what a wave issues");
  struct Frag { v4i k[KS]; };

  __shared__ v4i lds[2 * SLOT_V4];

  fetch_args(prm);
  const GemmArgs &g = prm.g;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wp = wave % WP, wq = wave / WP;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int NP = prm.swapped ? g.N : g.M, NQ = prm.swapped ? g.M : g.N;
  const int Kbytes = g.K * ESZ;
  const uint8_t *Pb = (const uint8_t *)(prm.swapped ? g.B : g.A), *Qb = (const uint8_t *)(prm.swapped ? g.A : g.B);
  const int64_t p_sb = (prm.swapped ? g.b_sb : g.a_sb) * ESZ, q_sb = (prm.swapped ? g.a_sb : g.b_sb) * ESZ;
  const int ldp = (int)(prm.swapped ? g.b_sj : g.a_si) * ESZ, ldq = (int)(prm.swapped ? g.a_si : g.b_sj) * ESZ;

  // This workgroup's run: tiles counted along Q, then P, then the batches; every XCD has a contiguous range of them (its
  // workgroups are blockIdx.x mod 8), shared out evenly over its workgroups.  Neighbours have neighbouring tiles of P at about the
  // same Q, so the lines that two tiles of D share (a pitch that is no multiple of 128 bytes) meet in the XCD's L2: runs along
  // P took 58 us for bf16 1000 x 1000 x 128, 64 batches, runs along Q take 51.
  const uint32_t total = (uint32_t)(prm.tiles_p * prm.tiles_q) * (uint32_t)g.batch, groups = (uint32_t)prm.groups >> 3;
  const uint32_t x = blockIdx.x & 7, lo = (uint32_t)((uint64_t)total * x >> 3), cnt = (uint32_t)((uint64_t)total * (x + 1) >> 3) - lo;
  ShortPos use;
  {
    const uint32_t j = blockIdx.x >> 3, at = (uint32_t)((uint64_t)cnt * j / groups), end = (uint32_t)((uint64_t)cnt * (j + 1) / groups);
    const uint32_t id = lo + at, row = id / (uint32_t)prm.tiles_q;
    use.q = __builtin_amdgcn_readfirstlane((int)(id - row * (uint32_t)prm.tiles_q));
    use.p = __builtin_amdgcn_readfirstlane((int)(row % (uint32_t)prm.tiles_p));
    use.bt = __builtin_amdgcn_readfirstlane((int)(row / (uint32_t)prm.tiles_p));
    use.left = __builtin_amdgcn_readfirstlane((int)(end - at));
    use.p_due = true;
  }
  const int drow = wave * 8 + lane / CPR;  // (passes advance by 32 rows: same swizzle)
  const int dcg = (lane % CPR) ^ swz(drow);
  // the lanes of the last chunk past the end of K read zeros; every instruction has lanes that are not (K is whole 16-byte pieces)
  const int oob_last = dcg * 16 < Kbytes - (NC - 1) * 128 ? 0 : (int)0x80000000;
  auto issue_panel = [&](const ShortPos &c, int slot) {
    const uint8_t *base = c.p_due ? Pb + p_sb * c.bt : Qb + q_sb * c.bt;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, 0x80000000, 0x00020000);
    const int row0 = c.p_due ? c.p * BP : c.q * BQ, last = (c.p_due ? NP : NQ) - 1, ld = c.p_due ? ldp : ldq;
    int voff[LD];
#pragma unroll
    for (int i = 0; i < LD; i++) voff[i] = min(row0 + drow + 32 * i, last) * ld + dcg * 16;
#pragma unroll
    for (int ch = 0; ch < NC; ch++)
#pragma unroll
      for (int i = 0; i < LD; i++)
        lds_dma16(rs, &lds[slot * SLOT_V4 + ch * CHUNK_V4 + (wave * 8 + 32 * i) * CPR], voff[i] | (ch == NC - 1 ? oob_last : 0), ch * 128);
  };

  // fragment addresses of even and odd 16-row tiles (gemm_mfma_pipe16.hpp)
  int frag_at[2][2];
#pragma unroll
  for (int par = 0; par < 2; par++)
#pragma unroll
    for (int kk = 0; kk < 2; kk++) frag_at[par][kk] = (par * 16 + r16) * CPR + ((2 * g4 + kk) ^ swz(par * 16 + r16));
  Frag pf[NC][TP], qf[NC][TQ];
  auto load_frags = [&](int slot, int row0, Frag (&f)[NC][4]) {
#pragma unroll
    for (int ch = 0; ch < NC; ch++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const v4i *base = &lds[slot * SLOT_V4 + ch * CHUNK_V4 + (row0 + (i >> 1) * 32) * CPR];
        f[ch][i].k[0] = base[frag_at[i & 1][0]];
        f[ch][i].k[1] = base[frag_at[i & 1][1]];
      }
  };
  static_assert(TP == 4 && TQ == 4, "64 x 64 per wave");

  // (the host sends only problems with one factor for all of D)
  const EpilogueScalars sc(g);
  const float scale = sc.alpha_s * sc.sa_s * sc.sb_s;
  ShortPos ask = use;  // the next panel to request
  int panels = 0;  // of those requested, not read yet
  for (int s = 0; s < 2; s++)
    if (ask.left > 0) { issue_panel(ask, s); short_advance(ask, prm.tiles_p, prm.tiles_q); panels++; }
  int slot = 0, st1 = 0, st2 = 0;  // stores that count, of the tile before and the one before that
  while (use.left > 0) {
    // wait for the panel; younger: st2, the next panel, st1
    switch (short_wait(SC, panels == 2, st1 + st2)) {
    case 0: asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(short_wait_n(SC, 0)) : "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(short_wait_n(SC, 1)) : "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(short_wait_n(SC, 2)) : "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(short_wait_n(SC, 3)) : "memory");
    }
    const ShortPos now = use;
    if (now.p_due) load_frags(slot, wp * WTP, pf);
    else load_frags(slot, wq * WTQ, qf);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    panels--;
    if (ask.left > 0) { issue_panel(ask, slot); short_advance(ask, prm.tiles_p, prm.tiles_q); panels++; }
    slot ^= 1;
    short_advance(use, prm.tiles_p, prm.tiles_q);
    st2 = st1;
    st1 = 0;
    if (now.p_due) continue;
    __builtin_amdgcn_sched_barrier(0);
    v4f acc[TP][TQ];
#pragma unroll
    for (int a = 0; a < TP; a++)
#pragma unroll
      for (int b = 0; b < TQ; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[a][b][v] = 0;
#pragma unroll
    for (int ch = 0; ch < NC; ch++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int a = 0; a < TP; a++)
#pragma unroll
          for (int b = 0; b < TQ; b++) {
            if constexpr (KIND == KIND_F16)
              acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, pf[ch][a].k[ks]), __builtin_bit_cast(v8h, qf[ch][b].k[ks]), acc[a][b], 0, 0, 0);
            else
              acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, pf[ch][a].k[ks]), __builtin_bit_cast(v8b, qf[ch][b].k[ks]), acc[a][b], 0, 0, 0);
          }
    const int p0 = now.p * BP, q0 = now.q * BQ;
    const int d_sq = (int)(prm.swapped ? g.d_si : g.d_sj), esz = g.d_type == CUDA_R_32F ? 4 : 2;  // (a pitch below kNarrowPitch: checked by the host)
    const int pc = p0 + wp * WTP, qc = q0 + wq * WTQ, p_left = NP - pc;
    const int64_t corner = (int64_t)qc * d_sq + pc;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((char *)g.D + (g.d_sb * now.bt + corner) * esz, 0,
                                                                        tile_window_bytes(d_sq, NP, NQ, corner, esz), 0x00020000);
#define ZLUDA_SHORT_STORE(DT_)                                              \
  if (p_left >= WTP) short_store<TP, TQ, DT_, false>(rs, d_sq, acc, scale, sc.sd, p_left); \
  else short_store<TP, TQ, DT_, true>(rs, d_sq, acc, scale, sc.sd, p_left);
    if (g.d_type == CUDA_R_16BF) { ZLUDA_SHORT_STORE(0) }
    else if (g.d_type == CUDA_R_16F) { ZLUDA_SHORT_STORE(1) }
    else { ZLUDA_SHORT_STORE(2) }
#undef ZLUDA_SHORT_STORE
    if (p0 + BP <= NP && q0 + BQ <= NQ) st1 = SC.stores;
  }
}

} // namespace zluda_amd
