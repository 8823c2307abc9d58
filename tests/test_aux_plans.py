"""Which plans carry an epilogue with an aux matrix in their own kernel: only grids that cover every tile of every batch, one workgroup each."""
import pytest

import planner_probe
from planner_probe import planned
from zluda_amd import abi as K

AUX, AUX_BIAS, DG, DG_SUMS = (K.CUBLASLT_EPILOGUE_GELU_AUX, K.CUBLASLT_EPILOGUE_GELU_AUX_BIAS, K.CUBLASLT_EPILOGUE_DGELU, K.CUBLASLT_EPILOGUE_DGELU_BGRAD)
H16, TR16 = K.ZLUDA_KERNEL_MFMA_H16, K.ZLUDA_KERNEL_MFMA_TR16


@pytest.mark.parametrize("epi", [AUX, DG, DG_SUMS])
@pytest.mark.parametrize("m,n,k,batch", [(2048, 4096, 128, 2), (4096, 2000, 64, 3), (512, 16384, 120, 9)])   # 512 tiles of 128 x 128 a batch
def test_walked_tiles_with_a_grid_of_one_batch(api, m, n, k, batch, epi):
    status, p, plan, keep = planned(api, m, n, k, batch, epi)
    assert status == 0 and (plan.kernel, plan.variant, plan.grid_x, plan.grid_y) == (H16, 3, 512, 1)
    assert planner_probe.aux_in_epilogue(p, plan) == 0


@pytest.mark.parametrize("epi", [AUX, AUX_BIAS, DG, DG_SUMS])
@pytest.mark.parametrize("cus", [64, 256])
def test_every_plan_that_carries_it_covers_the_batches(api, cus, epi):
    carried = 0
    for ta, tb in ((1, 0), (0, 0), (0, 1), (1, 1)):
        for m in (8, 64, 264, 1024, 2048):
            for n in (1, 65, 512, 2048):
                for k in (64, 128, 136, 2048):
                    for batch in (1, 2, 5, 8):
                        for family, variants in ((0, (-1,)), (H16, range(12)), (TR16, range(4))):
                            for v in variants:
                                status, p, plan, keep = planned(api, m, n, k, batch, epi, ta, tb, family=family, variant=v, cus=cus)
                                if status or planner_probe.aux_in_epilogue(p, plan) != 1:
                                    continue
                                carried += 1
                                if plan.kernel == H16 and plan.variant == 11:
                                    continue   # (the persistent kernel walks the batches itself)
                                assert plan.grid_y == batch and plan.grid_z == 1
                                if epi == DG_SUMS:
                                    assert plan.workspace >= planner_probe.aux_sum_bytes(p, plan)
    assert carried > 1000


def test_a_scale_of_d_keeps_the_pass_behind_the_persistent_kernel(api):
    status, p, plan, keep = planned(api, 4096, 4096, 2048, epi=AUX_BIAS)
    assert status == 0 and (plan.kernel, plan.variant) == (H16, 11)
    assert planner_probe.aux_in_epilogue(p, plan) == 1
    p.op.d_scale = planner_probe.BASE
    assert planner_probe.aux_in_epilogue(p, plan) == 0
