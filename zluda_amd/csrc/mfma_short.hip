// f16 and bf16 products of a short K and many tiles (kernels/gemm_mfma_short.hpp).
#include "kernels/gemm_mfma_short.hpp"
#include "mfma_launch.hpp"
namespace zluda_amd {
uint32_t launch_mfma_short(const MfmaParams &prm, bool bf16, uint32_t grid, hipStream_t s) {
  const dim3 gr(grid), bl(256);
  if (prm.g.K <= 64)
    return bf16 ? launch_kernel(gemm_mfma_short_kernel<KIND_BF16, 1>, gr, bl, s, prm) : launch_kernel(gemm_mfma_short_kernel<KIND_F16, 1>, gr, bl, s, prm);
  return bf16 ? launch_kernel(gemm_mfma_short_kernel<KIND_BF16, 2>, gr, bl, s, prm) : launch_kernel(gemm_mfma_short_kernel<KIND_F16, 2>, gr, bl, s, prm);
}
} // namespace zluda_amd
