// f16 instantiations of the K-contiguous MFMA kernels with the epilogues that keep or use the GELU input.
#include "mfma_launch.hpp"
namespace zluda_amd {
uint32_t launch_mfma_aux_f16(const MfmaParams &prm, const zluda_gemm_plan &plan, hipStream_t s) {
  return launch_mfma_variant<KIND_F16, 0, 0, true>(prm, plan, s);
}
} // namespace zluda_amd
