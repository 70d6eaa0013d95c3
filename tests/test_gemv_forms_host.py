"""How a linear of one row streams its weights (csrc/gemm.hip: gemv2_form), asked of the library on the host.  Cases of one row a wave were timed with two and with four loads of it on the way."""
import ctypes

import pytest


def _form(N, K, act=0, norm=0):
    from llava_mi355x import _C
    f = (ctypes.c_int32 * 2)()
    _C.check(_C.lib.lmx_op_gemv_form(N, K, act, norm, f))
    return tuple(f)


@pytest.mark.parametrize("N,K,ahead", [(8192, 512, 2), (12288, 512, 2), (8192, 1024, 2), (256, 768, 2), (1024, 1032, 4), (2048, 1152, 4), (2048, 2048, 4), (2056, 2048, 2), (5120, 2048, 2), (6144, 1792, 2),
                                       (8192, 1408, 2), (11768, 1408, 2), (11776, 1408, 4), (12288, 2048, 4), (5120, 2056, 4), (2048, 5632, 4), (2048, 7680, 4), (4096, 4096, 4), (2048, 8192, 8)])
def test_loads_of_a_row_ahead(N, K, ahead):
    assert _form(N, K) == (1, ahead)


def test_two_rows_a_wave():
    assert _form(4096, 4096, norm=1) == (2, 4) and _form(8200, 4096) == (2, 4) and _form(1024, 512, act=3) == (2, 4) and _form(22016, 4096, act=3) == (2, 4)
