// MXFP4 instantiations of the slab decode kernel (v_mfma_scale_f32_16x16x128_f8f6f4 with FP4 operands).
#include "decode_launch.hpp"
namespace zluda_amd {
uint32_t launch_decode_slab_mx(const DecodeParams &prm, const zluda_gemm_plan &plan, int nb, hipStream_t s) {
  return launch_decode_slab<KIND_MXF4>(prm, plan, nb, s);
}
} // namespace zluda_amd
