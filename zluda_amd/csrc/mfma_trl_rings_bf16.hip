// bf16 instantiations of gemm_mfma_pipe16_kernel for operands with unit stride along their row index: the small tiles, on rings of their own.
#include "mfma_tr_launch.hpp"
namespace zluda_amd {
uint32_t launch_trl_rings_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s) {
  return launch_trl_rings<KIND_BF16>(prm, plan, pkc, qkc, s);
}
} // namespace zluda_amd
