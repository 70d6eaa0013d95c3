"""How a linear of one row streams its weights (csrc/gemm.hip: gemv2_form, gemv2_res_form, gemv_heads_splits), asked of the library on the host.  Cases of one row a wave were timed with two and with four loads of it on the way."""
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


@pytest.mark.parametrize("N,K,act,form", [(2552, 2048, 0, (1, 4, 8)), (2560, 2048, 0, (2, 2, 8)), (4096, 2048, 0, (2, 2, 8)), (4104, 2048, 0, (2, 4, 4)), (6144, 2048, 0, (2, 4, 4)), (6152, 2048, 0, (2, 2, 8)),
                                          (5120, 1536, 0, (2, 2, 8)), (5120, 2056, 0, (2, 2, 8)), (5632, 2048, 3, (2, 4, 4)), (11264, 2048, 3, (2, 2, 8)), (2496, 2048, 3, (2, 4, 4)),
                                          (4096, 4096, 0, (1, 4, 8)), (6144, 4096, 0, (2, 2, 8)), (4088, 4096, 0, (2, 4, 4)), (8192, 4104, 0, (2, 4, 4))])
def test_a_row_formed_in_front(N, K, act, form):
    """Eight waves share the row where that takes less time than four."""
    from llava_mi355x import _C
    f = (ctypes.c_int32 * 3)()
    _C.check(_C.lib.lmx_op_gemv_residual_form(N, K, act, f))
    assert tuple(f) == form


def test_splits_that_the_projection_takes():
    from llava_mi355x import _C

    def most(dt, N, heads, D):
        s = ctypes.c_int32(-1)
        _C.check(_C.lib.lmx_op_gemv_heads_splits(dt, N, heads, D, s))
        return s.value
    for dt in (_C.DTYPE_BF16, _C.DTYPE_F16):
        assert [most(dt, 2056, h, 128) for h in (1, 8, 16, 17, 24, 32, 33)] == [16, 16, 16, 15, 10, 8, 0]
    assert most(_C.DTYPE_F32, 2056, 8, 128) == 0
