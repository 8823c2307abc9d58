// Launchers of the transposing MFMA kernel (kernels/gemm_mfma_tr.hpp); one translation unit per
// element kind so that the template instantiations compile in parallel.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels/gemm_mfma_pipe16.hpp"
#include "kernels/gemm_mfma_tr.hpp"
#include "launch_util.hpp"
#include "planner.hpp"

namespace zluda_amd {

// plan.variant indexes kTrVariants (planner.hpp); pkc / qkc: operand P / Q has unit stride along K.  AUX: the epilogues with an aux
// matrix, on the variants that have them (aux_in_epilogue()).
template <int KIND, int FQ, int FP, bool AUX = false>
inline uint32_t launch_tr_variant(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s) {
  const dim3 grid(plan.grid_x, plan.grid_y, plan.grid_z > 1 ? plan.grid_z : 1);  // z: split-K shares
#define ZLUDA_TR_MODE(BP, BQ, WP, WQ, PK, QK)                                                                   \
  if (pkc == PK && qkc == QK) {                                                                                 \
    return launch_kernel(gemm_mfma_tr_kernel<KIND, FQ, FP, BP, BQ, WP, WQ, PK, QK, false, 1, AUX>, grid, dim3(WP * WQ * 64), s, prm); \
  }
#define ZLUDA_TR_CASE(V, BP, BQ, WP, WQ)                                                                        \
  case V:                                                                                                       \
    static_assert(kTrVariants[V].bp == BP && kTrVariants[V].bq == BQ && kTrVariants[V].wp == WP &&              \
                  kTrVariants[V].wq == WQ && !kTrVariants[V].m16, "variant table mismatch");                                           \
    if constexpr (!AUX || aux_on_wave_tile32(BP / WP, BQ / WQ)) {                                               \
      ZLUDA_TR_MODE(BP, BQ, WP, WQ, false, false) ZLUDA_TR_MODE(BP, BQ, WP, WQ, false, true)                    \
      ZLUDA_TR_MODE(BP, BQ, WP, WQ, true, false) ZLUDA_TR_MODE(BP, BQ, WP, WQ, true, true)                      \
    }                                                                                                           \
    break;
#define ZLUDA_TR_KG(V, BP, BQ, PK, QK)                                                                            \
  if (plan.variant == V && pkc == PK && qkc == QK)                                                               \
    return launch_kernel(gemm_mfma_tr_kernel<KIND, FQ, FP, BP, BQ, 2, 2, PK, QK, false, 2, AUX>, grid, dim3(512), s, prm);
  if (plan.block == 512 && (plan.variant == 1 || plan.variant == 2)) {  // (tr_two_k_groups())
    if constexpr (kind_is_h16(KIND)) {
      ZLUDA_TR_KG(1, 128, 128, false, false) ZLUDA_TR_KG(1, 128, 128, false, true) ZLUDA_TR_KG(1, 128, 128, true, false) ZLUDA_TR_KG(1, 128, 128, true, true)
      ZLUDA_TR_KG(2, 64, 64, false, false) ZLUDA_TR_KG(2, 64, 64, false, true) ZLUDA_TR_KG(2, 64, 64, true, false) ZLUDA_TR_KG(2, 64, 64, true, true)
    }
    return CUBLAS_STATUS_INVALID_VALUE;
  }
#undef ZLUDA_TR_KG
  switch (plan.variant) {
    ZLUDA_TR_CASE(0, 256, 256, 2, 4)
    ZLUDA_TR_CASE(1, 128, 128, 2, 2)
    ZLUDA_TR_CASE(2, 64, 64, 2, 2)
  case 3:  // variant 0's tile on the 16x16 MFMA shape (int8, f16, bf16)
    static_assert(kTrVariants[3].bp == 256 && kTrVariants[3].bq == 256 && kTrVariants[3].wp == 2 && kTrVariants[3].wq == 4 &&
                  kTrVariants[3].m16, "variant table mismatch");
    if constexpr (KIND == KIND_I8 || kind_is_h16(KIND)) {
#define ZLUDA_TR16_MODE(PK, QK)                                                                                  \
  if (pkc == PK && qkc == QK)                                                                                    \
    return launch_kernel(gemm_mfma_tr_kernel<KIND, FQ, FP, 256, 256, 2, 4, PK, QK, true, 1, AUX>, grid, dim3(512), s, prm);
      ZLUDA_TR16_MODE(false, false) ZLUDA_TR16_MODE(false, true) ZLUDA_TR16_MODE(true, false) ZLUDA_TR16_MODE(true, true)
#undef ZLUDA_TR16_MODE
    }
    break;
  default: break;
  }
#undef ZLUDA_TR_CASE
#undef ZLUDA_TR_MODE
  return CUBLAS_STATUS_INVALID_VALUE;
}

// the variants 1, 2 and 3 where tr_lds_reads() says so: their grids, with the transposition in the LDS reads
uint32_t launch_trl_f16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_trl_rings_f16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_trl_rings_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_trl_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
// (a problem whose `act` is an epilogue with an aux matrix)
uint32_t launch_trl_aux_f16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_trl_aux_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_aux_f16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_aux_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_i8(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_f8(const MfmaParams &prm, const zluda_gemm_plan &plan, int fq, int fp, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_f8_e5m2q(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_f8_e5m2p(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_f16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);
uint32_t launch_tr_f32(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s);

// Which of the two below: the variant 2, and the variant 1 on its deep ring.  Their kernels have a translation unit, i.e. a code object, of their
// own (mfma_trl_rings_*.hip): in one with them the 256 x 256 tiles took 1 to 2 % longer (bf16 4096 x 4096 x 256 A:N B:N, same code).
inline bool trl_on_rings(const zluda_gemm_plan &plan) {
  return plan.variant == 2 || tr_ring_stages((int)plan.variant, (uint64_t)plan.grid_x * plan.grid_y * (plan.grid_z > 1 ? plan.grid_z : 1), zluda_gemm_device_cu_count()) > 2;
}

template <int KIND, bool AUX = false>
inline uint32_t launch_trl_rings(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s) {
  const dim3 grid(plan.grid_x, plan.grid_y, plan.grid_z > 1 ? plan.grid_z : 1);
  const int stages = tr_ring_stages((int)plan.variant, (uint64_t)grid.x * grid.y * grid.z, zluda_gemm_device_cu_count());
  if (plan.variant == 2) {
    // 17 KiB a stage: as many of them as the workgroups that share a CU have room for.  (64 x 64 tiles, bf16, us from memory and from the caches,
    // transposed in registers before: 704 x 1000 x 2104, 176 workgroups 17.9 -> 14.2 and 13.5 -> 10.6; 2104 x 704 x 1000, 363, 16.9 -> 13.8 and 11.9 -> 10.7.)
#define ZLUDA_TRL_64(PK, QK, NS)                                                                                      \
  if (pkc == PK && qkc == QK)                                                                                        \
    return launch_kernel(gemm_mfma_pipe16_kernel<KIND, 0, 0, 64, 64, 2, 2, !PK, !QK, NS, AUX>, grid, dim3(256), s, prm);
#define ZLUDA_TRL_64_RING(NS) { ZLUDA_TRL_64(false, false, NS) ZLUDA_TRL_64(false, true, NS) ZLUDA_TRL_64(true, false, NS) }
    if (stages == kTr64Stages[0]) ZLUDA_TRL_64_RING(kTr64Stages[0])
    else if (stages == kTr64Stages[1]) ZLUDA_TRL_64_RING(kTr64Stages[1])
    else ZLUDA_TRL_64_RING(kTr64Stages[2])
#undef ZLUDA_TRL_64_RING
#undef ZLUDA_TRL_64
    return CUBLAS_STATUS_INVALID_VALUE;
  }
  // One workgroup to a CU: four stages of 33 KiB instead of two, all but the one that is multiplied on their way (a stage's time is far
  // below a round trip to memory; with two workgroups the other one fills the gaps, and two rings of four do not fit).  bf16, us from
  // memory and from the caches: 2048^3 A:N B:N 34.2 -> 25.0 and 28.4 -> 21.3, A:N B:T 33.0 -> 25.0 and 29.3 -> 21.3, 1024 x 4096 x 4096 61.1 -> 41.7 and
  // 46.9 -> 34.4; at 11 stages 2048 x 2048 x 704 14.0 -> 12.6 and level; on 512 tiles 2048 x 4096 x 8192 132 -> 165, 4096 x 2048 x 512 15 -> 20.
  if (plan.variant == 1 && stages == kTrDeepStages) {
#define ZLUDA_TRL_DEEP(PK, QK)                                                                                        \
  if (pkc == PK && qkc == QK)                                                                                        \
    return launch_kernel(gemm_mfma_pipe16_kernel<KIND, 0, 0, 128, 128, 2, 2, !PK, !QK, kTrDeepStages, AUX>, grid, dim3(256), s, prm);
    ZLUDA_TRL_DEEP(false, false) ZLUDA_TRL_DEEP(false, true) ZLUDA_TRL_DEEP(true, false)
#undef ZLUDA_TRL_DEEP
  }
  return CUBLAS_STATUS_INVALID_VALUE;
}

template <int KIND, bool AUX = false>
inline uint32_t launch_trl(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s) {
  const dim3 grid(plan.grid_x, plan.grid_y, plan.grid_z > 1 ? plan.grid_z : 1);
#define ZLUDA_TRL_MODE(BP, BQ, WP, WQ, PK, QK)                                                                       \
  if (pkc == PK && qkc == QK)                                                                                        \
    return launch_kernel(gemm_mfma_pipe16_kernel<KIND, 0, 0, BP, BQ, WP, WQ, !PK, !QK, 2, AUX>, grid, dim3(WP * WQ * 64), s, prm);
#define ZLUDA_TRL_CASE(V, BP, BQ, WP, WQ)                                                                            \
  case V:                                                                                                            \
    static_assert(kTrVariants[V].bp == BP && kTrVariants[V].bq == BQ && kTrVariants[V].wp == WP &&                   \
                  kTrVariants[V].wq == WQ, "variant table mismatch");                                                \
    ZLUDA_TRL_MODE(BP, BQ, WP, WQ, false, false) ZLUDA_TRL_MODE(BP, BQ, WP, WQ, false, true)                         \
    ZLUDA_TRL_MODE(BP, BQ, WP, WQ, true, false)                                                                      \
    break;
  switch (plan.variant) {
    ZLUDA_TRL_CASE(1, 128, 128, 2, 2)
    ZLUDA_TRL_CASE(3, 256, 256, 2, 4)
  default: break;
  }
#undef ZLUDA_TRL_CASE
#undef ZLUDA_TRL_MODE
  return CUBLAS_STATUS_INVALID_VALUE;
}

} // namespace zluda_amd
