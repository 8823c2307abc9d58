// bf16 instantiations of the transposing MFMA kernel with the epilogues that keep or use the GELU input.
#include "mfma_tr_launch.hpp"
namespace zluda_amd {
uint32_t launch_tr_aux_bf16(const MfmaParams &prm, const zluda_gemm_plan &plan, bool pkc, bool qkc, hipStream_t s) {
  return launch_tr_variant<KIND_BF16, 0, 0, true>(prm, plan, pkc, qkc, s);
}
} // namespace zluda_amd
