"""The rules by which kernels are chosen, asked on the host: no GPU is needed to ask."""
import pytest
import torch

from tessweave_engine_amd.kernels import ops
from tessweave_engine_amd.kernels.lib import library

F32, BF16 = 0, 1


@pytest.mark.parametrize("m,n,k,ranges", [(489, 5496, 4736, 2), (1900, 3584, 18944, 2), (536, 5120, 13824, 4)])
def test_products_that_one_kernel_does_not_take_keep_the_plan_of_the_other(m, n, k, ranges):
    """Four columns more than a multiple of 8: results are not rows of 16 bytes, so that the tiles whose waves take turns do not run,
    and the K ranges are those of the tiles that do. The scratch holds either plan's."""
    lib = library()
    assert lib.tw_linear_partial_splits_rows(BF16, 1, m, n + 4, k, k) == ranges
    assert lib.tw_linear_workspace_bytes(BF16, m, n + 4, k) >= ranges * m * (n + 4) * 4
    for cols in (n, n + 4):
        named = lib.tw_linear_partial_splits_rows(BF16, 1, m, cols, k, k)
        assert lib.tw_linear_workspace_bytes(BF16, m, cols, k) >= named * m * cols * 4


@pytest.mark.parametrize("dtype,m,n,k,whole", [(BF16, 8, 2048, 2304, True), (BF16, 8, 2304, 2560, False), (BF16, 8, 2304, 2816, True), (BF16, 1, 2304, 3584, False),
                                               (BF16, 8, 2560, 3584, True), (BF16, 9, 2560, 3584, False), (F32, 8, 2560, 1536, False), (F32, 8, 2560, 1792, True),
                                               (F32, 1, 2560, 2304, False), (F32, 8, 3072, 2816, True), (F32, 8, 3072, 3328, False), (F32, 8, 3584, 3584, True),
                                               (F32, 8, 3584, 3328, False), (F32, 9, 3584, 2048, False)])
def test_sums_for_the_next_kernel_over_the_whole_of_k(dtype, m, n, k, whole):
    """Up to 8 rows and a long K: K ranges stay where they are the faster form, one workgroup a CU of whole stages."""
    assert (library().tw_linear_partial_splits_rows(dtype, 1, m, n, k, k) == 1) == whole


@pytest.mark.parametrize("rows", [1, 8])
def test_an_activation_behind_few_rows_asks_for_what_its_kernel_takes(rows):
    """Rows 2,050 elements apart are no multiple of 16 bytes apart, which the kernel refuses of a single row too."""
    weight = ops.shuffle_weight(torch.zeros(4096, 2048, dtype=torch.bfloat16))
    assert ops.linear_act_few_pays(torch.zeros(rows, 2048, dtype=torch.bfloat16), weight)
    assert ops.linear_act_few_pays(torch.zeros(rows + 1, 2056, dtype=torch.bfloat16)[:rows, :2048], weight)
    assert not ops.linear_act_few_pays(torch.zeros(rows + 1, 2050, dtype=torch.bfloat16)[:rows, :2048], weight)
