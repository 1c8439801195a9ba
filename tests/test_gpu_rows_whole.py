"""The streaming kernel with its rows whole in LDS (blkq4_skinny.hip).  The library's own choice does not take it, a plan by name
(blkq4_gemm_with_plan_sm80) starts it: every shape that exists, in both blockings and both types, against the reference's exact
construction (test/blkq4_fp16_gemm_sm80_test.cu:194-256,469-472), bit for bit."""

import pytest

from test_gpu_gemm import check_plans_exact

pytestmark = pytest.mark.gpu

# up to 16 rows: eight, sixteen and four waves that split K, four waves with column tiles of their own
FEW_ROWS = [f"streaming 4 {nt} 1 8 1 8" for nt in (1, 2, 3)] + ["streaming 2 1 1 8 1 8", "streaming 8 1 1 4 1 4"] + \
           [f"streaming 2 {nt} 1 16 1 16" for nt in (1, 2, 3)] + [f"streaming 4 {nt} 1 4 1 4" for nt in (1, 2, 3)] + ["streaming 4 1 1 4 1 1"]
ROW_GROUPS = [f"streaming 2 {nt} 2 8 1 8" for nt in (1, 2, 4, 6, 8)]


def _along_n(plans):
    return [plan for plan in plans if plan.split()[2] == "1"]   # one column tile only


@pytest.mark.parametrize("bs,has_offsets,m,n,k", [
    # one slice for all waves; a last slice of two units (K = 64 mod 128); columns that end inside a workgroup's; waves that ask
    # for more slices than they have
    (64, True, 1, 64, 64), (16, False, 9, 352, 576), (32, True, 16, 224, 2112), (32, False, 4, 544, 448), (64, False, 2, 192, 4288),
    (64, True, 17, 192, 64), (32, False, 40, 352, 576), (16, True, 97, 224, 1088), (64, False, 32, 128, 2048)])
@pytest.mark.parametrize("column_wise", [True, False])
@pytest.mark.parametrize("bf16", [False, True])
def test_every_shape_of_workgroup_is_exact(oracle, capi, device, bs, has_offsets, m, n, k, column_wise, bf16):
    plans = FEW_ROWS if m <= 16 else ROW_GROUPS
    check_plans_exact(oracle, capi, device, bs, has_offsets, column_wise, m, n, k, plans if column_wise else _along_n(plans), bf16)


@pytest.mark.parametrize("bs,has_offsets,column_wise,m,n,k,bf16,plans", [
    # workgroups that walk over several column groups: from twice as many on as there are resident workgroups (256, one per
    # compute unit, where the rows and the partial tiles take more than half of LDS), shared out over the row groups
    (64, True, True, 16, 8224, 4288, False, _along_n(FEW_ROWS)), (32, False, False, 16, 8224, 4288, True, _along_n(FEW_ROWS)),
    (32, False, True, 16, 16448, 4096, True, ["streaming 4 2 1 8 1 8", "streaming 4 2 1 4 1 4"]),
    (16, True, True, 16, 24608, 4096, False, ["streaming 4 3 1 8 1 8", "streaming 4 3 1 4 1 4"]),
    (64, True, True, 97, 2080, 1088, True, ROW_GROUPS[:1]), (64, True, False, 97, 2112, 1088, False, ROW_GROUPS[:1]),
    (32, True, False, 97, 2080, 1088, True, ROW_GROUPS[:1]), (32, False, True, 97, 4128, 1088, False, ROW_GROUPS[1:2]),
    (16, True, True, 97, 8224, 1088, True, ROW_GROUPS[2:3]), (64, False, True, 97, 12320, 960, False, ROW_GROUPS[3:4]),
    (32, True, True, 97, 16416, 448, True, ROW_GROUPS[4:]),
    # and those with column tiles of their own, 64 columns a workgroup
    (64, True, True, 16, 32832, 4288, False, ["streaming 4 1 1 4 1 1"])])
def test_workgroups_that_walk_over_column_groups_are_exact(oracle, capi, device, bs, has_offsets, column_wise, m, n, k, bf16, plans):
    check_plans_exact(oracle, capi, device, bs, has_offsets, column_wise, m, n, k, plans, bf16)
