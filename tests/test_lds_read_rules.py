"""Which form of the transposing family's 64 x 64 tile runs 16-byte aligned 16-bit operands: transposed by the LDS reads, but in registers for
a K of one stage there and for a long operand along its row index beside a few K-contiguous tokens on four to six workgroups per CU."""
import pytest

import planner_probe
from planner_probe import planned
from zluda_amd import abi as K

TR16 = K.ZLUDA_KERNEL_MFMA_TR16


@pytest.mark.parametrize("m,n,k,ta,tb,lds", [
    (65536, 16, 512, 0, 0, 0), (16, 65536, 512, 1, 1, 0),      # 1024 workgroups, either operand the long one
    (65536, 16, 512, 0, 1, 1), (65536, 16, 512, 1, 1, 1),      # both along their row index; the long one K-contiguous
    (65536, 16, 72, 0, 0, 1), (65536, 17, 512, 0, 0, 1),
    (49152, 16, 512, 0, 0, 1), (49160, 16, 512, 0, 0, 0),      # three workgroups per CU, and more
    (98304, 16, 512, 0, 0, 0), (98312, 16, 512, 0, 0, 1),      # six, and more
    (1024, 1024, 512, 0, 0, 1), (1024, 1024, 32, 0, 1, 0), (1024, 1024, 40, 0, 1, 1), (1024, 1024, 64, 0, 0, 0), (1024, 1024, 72, 1, 1, 1)])
def test_sixty_four_square(api, m, n, k, ta, tb, lds):
    status, p, plan, keep = planned(api, m, n, k, ta=ta, tb=tb, workspace=0, family=TR16, variant=2)
    assert status == 0 and plan.grid_z == 1
    assert planner_probe.lds_reads(p, plan, 256) == lds and plan.block == 256


def test_shares_of_k_count(api):
    status, p, plan, keep = planned(api, 14336, 16, 4096, ta=0, workspace=32 << 20, family=TR16)
    assert status == 0 and (plan.variant, plan.grid_x, plan.grid_z) == (2, 224, 4)
    assert planner_probe.lds_reads(p, plan, 256) == 0
    status, p, plan, keep = planned(api, 14336, 16, 4096, ta=0, workspace=0, family=TR16, variant=2)
    assert planner_probe.lds_reads(p, plan, 256) == 1


# LDS of a CU: 132 KiB of a ring of four stages of 128 x 128 tiles, 66 of two; 99, 50 and 33 of 64 x 64 tiles on six, three and two; in registers four
# workgroups
@pytest.mark.parametrize("m,n,k,ta,tb,variant,per_cu", [
    (2048, 2048, 2048, 0, 0, 1, 1), (2048, 2176, 2048, 0, 0, 1, 2), (1024, 1024, 1024, 0, 1, 2, 1), (1024, 1088, 1024, 0, 1, 2, 3),
    (4096, 1024, 1024, 0, 1, 2, 4), (65536, 16, 512, 0, 0, 2, 4), (2048, 2048, 128, 0, 0, 1, 4), (2044, 2048, 512, 0, 0, 1, 4), (4096, 4096, 512, 0, 0, 3, 1)])
def test_waves_are_those_of_the_form_that_runs(api, m, n, k, ta, tb, variant, per_cu):
    status, p, plan, keep = planned(api, m, n, k, ta=ta, tb=tb, workspace=0, family=TR16, variant=variant)
    assert status == 0 and plan.waves == pytest.approx(plan.grid_x / (256 * per_cu))
