"""How a grouped product of few rows a group reads its weights (csrc/moe.hip: group_gemm_form), asked of the library on the host.  Every case was timed in both forms."""
import ctypes

import pytest


def _form(rows, groups, N, K, bm, planned=1):
    from llava_mi355x import _C
    f = (ctypes.c_int32 * 2)()
    _C.check(_C.lib.lmx_op_group_gemm_form(rows, groups, planned, N, K, bm, f))
    return bool(f[0]), f[1]


# rows of all groups, groups, N, K, tile rows -> streaming, slabs
CASES = [((32, 4, 704, 6528, 32), (False, 4)), ((54, 6, 576, 6144, 32), (False, 4)), ((40, 4, 1920, 3776, 32), (False, 4)), ((128, 16, 960, 896, 32), (False, 4)), ((88, 4, 2560, 2304, 32), (False, 4)),
         ((64, 4, 3328, 1024, 32), (False, 4)), ((64, 8, 3072, 4096, 32), (True, 4)), ((64, 8, 3072, 4032, 32), (False, 4)), ((128, 16, 1792, 704, 32), (True, 4)), ((128, 16, 1664, 704, 32), (False, 4)),
         ((128, 16, 4096, 2752, 32), (True, 4)), ((128, 16, 4224, 1024, 32), (True, 2)), ((128, 16, 5504, 4096, 32), (True, 2)), ((128, 16, 8192, 1024, 32), (True, 2)),
         ((128, 16, 8320, 704, 32), (True, 4)), ((144, 16, 10176, 2176, 32), (True, 4)), ((160, 8, 5056, 3840, 32), (True, 4)), ((409, 16, 5504, 4096, 32), (True, 2)), ((410, 16, 5504, 4096, 32), (False, 4)),
         ((480, 16, 5504, 4096, 64), (True, 3)), ((819, 16, 5504, 4096, 64), (True, 3)), ((820, 16, 5504, 4096, 64), (False, 3)), ((240, 8, 576, 2240, 64), (False, 3))]


@pytest.mark.parametrize("case,form", CASES)
def test_weights_of_a_mixture(case, form):
    assert _form(*case) == form


@pytest.mark.parametrize("rows,groups,N,form", [(32, 32, 512, (False, 4)), (32, 32, 896, (True, 4)), (33, 32, 896, (False, 4)), (4, 16, 128, (False, 4)), (8, 64, 1408, (True, 4))])
def test_weights_of_heads(rows, groups, N, form):
    """Without a plan every group has the same rows; never two slabs."""
    assert _form(rows, groups, N, 512, 32, planned=0) == form
