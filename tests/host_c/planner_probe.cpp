// The planner's decisions that no plan names, for tests: built as a shared library of its own (planner.cpp needs no device).
#include "../../zluda_amd/csrc/planner.cpp"

#define PROBE extern "C" __attribute__((visibility("default")))

// whether the kernel of `plan` carries the aux epilogue of `p` itself, as launch_planned() asks; -1: not a valid problem
PROBE int probe_aux_in_epilogue(const zluda_gemm_problem *p, const zluda_gemm_plan *plan) {
  Lowered l;
  return lower_problem(p, false, &l) ? -1 : aux_in_epilogue(l, *plan, false);
}
// bytes of the partial sums that it then writes for DGELU_BGRAD
PROBE uint64_t probe_aux_sum_bytes(const zluda_gemm_problem *p, const zluda_gemm_plan *plan) {
  Lowered l;
  return lower_problem(p, false, &l) ? 0 : (uint64_t)aux_sum_shares(l, *plan) * l.g.M * l.g.batch * 4;
}
// whether the transposing kernel of `plan` does so by its LDS reads, as launch_tr() asks
PROBE int probe_lds_reads(const zluda_gemm_problem *p, const zluda_gemm_plan *plan, uint32_t cus) {
  Lowered l;
  if (lower_problem(p, false, &l)) return -1;
  return tr_lds_reads(l, (int)plan->variant, (uint64_t)plan->grid_x * plan->grid_y * std::max(plan->grid_z, 1u), plan->grid_z, cus);
}
PROBE uint32_t probe_plan(const zluda_gemm_problem *p, uint32_t kernel, int32_t variant, uint32_t cus, zluda_gemm_plan *plan) {
  return zluda_gemm_plan_problem(p, kernel, variant, cus, plan);
}
