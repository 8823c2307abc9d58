// bf16 instantiations of gemm_mfma_pipe16_kernel for operands with unit stride along their row index, with the epilogues that keep or
// use the GELU input.
#include "mfma_tr_launch.hpp"
namespace zluda_amd {
uint32_t launch_trl_aux_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s) {
  return trl_on_rings(plan) ? launch_trl_rings<KIND_BF16, true>(prm, plan, pkc, qkc, s) : launch_trl<KIND_BF16, true>(prm, plan, pkc, qkc, s);
}
} // namespace zluda_amd
