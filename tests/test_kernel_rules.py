"""The rules by which kernels are chosen, asked on the host: no GPU is needed to ask."""
import pytest

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
