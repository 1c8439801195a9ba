"""The streaming kernel with rows staged slice by slice (blkq4_staged.hip), every shape of workgroup asked for by name: the
reference's exact construction (test/blkq4_fp16_gemm_sm80_test.cu:194-256,469-472) comes out bit for bit where the kernel
can go wrong -- fewer 64-deep slices than waves, a slice count that leaves some waves a round more, columns that end inside
a workgroup's, row groups that are not full."""

import pytest
import torch

from test_gpu_gemm import bits_of, check_plans_exact, exact_problem

pytestmark = pytest.mark.gpu

ROW_GROUPS = [f"streaming 2 {nt} 2 8 2 8" for nt in (1, 2, 4, 6, 8)]
FEW_ROWS = [f"streaming 2 {nt} 1 {waves} 2 {waves}" for nt in (4, 5, 6, 7) for waves in (4, 8)] + \
           [f"streaming 4 {nt} 1 8 2 8" for nt in (1, 2, 3)]

CASES = [
    # block size, zero-points, rows, columns, K.  One slice for eight waves; 33 and 67 slices: the older waves' extra rounds
    (64, True, 17, 32, 64), (16, True, 33, 352, 2112), (32, False, 48, 224, 4288), (64, False, 25, 544, 576),
    # groups of 8 rows and less, of more than 24, the last row group short
    (32, True, 40, 96, 128), (16, False, 64, 128, 1024), (64, True, 129, 288, 320),
    # up to 16 rows
    (64, True, 1, 32, 64), (16, True, 16, 352, 2112), (32, False, 9, 224, 4288), (64, False, 8, 544, 576), (32, True, 5, 96, 192),
]


@pytest.mark.parametrize("bs,has_offsets,m,n,k", CASES)
@pytest.mark.parametrize("bf16", [False, True])
def test_every_shape_of_workgroup_is_exact(oracle, capi, device, bs, has_offsets, m, n, k, bf16):
    check_plans_exact(oracle, capi, device, bs, has_offsets, True, m, n, k, ROW_GROUPS if m > 16 else FEW_ROWS + ROW_GROUPS[:2], bf16)


@pytest.mark.parametrize("bs,has_offsets,m,n,k", [
    (64, True, 17, 64, 64), (16, False, 33, 352, 2112), (32, True, 48, 224, 576), (32, False, 1, 96, 64), (64, False, 9, 192, 4288),
    (16, True, 16, 48 * 16, 128),
])
@pytest.mark.parametrize("bf16", [False, True])
def test_blocks_along_n_are_exact(oracle, capi, device, bs, has_offsets, m, n, k, bf16):
    plans = ["streaming 2 1 2 8 2 8"] if m > 16 else ["streaming 4 1 1 8 2 8", "streaming 2 1 2 8 2 8"]
    check_plans_exact(oracle, capi, device, bs, has_offsets, False, m, n, k, plans, bf16)


@pytest.mark.parametrize("bs,has_offsets,m,n,k,bf16", [(64, True, 48, 11008, 4096, False), (32, True, 12, 4096, 11008, True)])
def test_as_the_library_chooses_it_with_a_bias_and_the_same_bits_every_time(oracle, capi, device, bs, has_offsets, m, n, k, bf16):
    text = capi.gemm_plan(bs, True, m, n, k, has_offsets, bf16)[2]
    assert text.startswith("streaming:") and "rows staged per slice" in text, text
    a_dev, q_w, q_s, q_zp, ref = exact_problem(oracle, capi, device, bs, has_offsets, True, m, n, k, bf16)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 0.5).to(a_dev.dtype).to(device)
    want = torch.from_numpy(ref.view("int16").copy()).to(device).view(a_dev.dtype)
    noise = torch.randn(m, k, generator=torch.Generator().manual_seed(k)).to(a_dev.dtype).to(device)
    first = None
    for _ in range(3):
        out = torch.full((m, n), float("nan"), dtype=a_dev.dtype, device=device)
        capi.gemm(bs, True, m, n, k, a_dev, q_w, q_s, q_zp, out, bias=bias, bf16=bf16)
        torch.cuda.synchronize()
        assert (bits_of(out) == bits_of(want + bias)).all()   # (rounded before and after)
        capi.gemm(bs, True, m, n, k, noise, q_w, q_s, q_zp, out, bf16=bf16)
        torch.cuda.synchronize()
        first = bits_of(out) if first is None else first
        assert (bits_of(out) == first).all()   # the waves' partial sums are added in wave order
