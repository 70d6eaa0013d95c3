"""Which linears of one token share a launch with the work beside them, asked of the library on the host.  Every case was timed both ways: the shared launch is taken where it is the shorter
one (csrc/delta.hip: delta_decode_joins, csrc/moe.hip: group_gemv_joins)."""
import ctypes

import pytest
import torch


def _delta(heads, dim, N, K, dt=torch.bfloat16):
    from llava_mi355x import _C
    f = ctypes.c_int32()
    _C.check(_C.lib.lmx_op_delta_joins(_C.torch_dtype_code(dt), heads, dim, N, K, f))
    return bool(f.value)


# heads, head width, gate | up rows, width
TOGETHER = [(8, 128, 1024, 1024), (8, 128, 32768, 1024), (16, 128, 11264, 2048), (16, 128, 22016, 2048), (32, 64, 22016, 2048), (24, 128, 1024, 3072), (24, 128, 22016, 3072), (28, 128, 32768, 3584),
            (32, 128, 8192, 4096), (32, 128, 11264, 4096), (64, 64, 11264, 4096), (36, 128, 18432, 4608), (40, 128, 22016, 5120), (48, 128, 14336, 6144), (48, 128, 8192, 6144),
            (56, 128, 14336, 7168), (64, 128, 8192, 8192), (64, 128, 11264, 8192), (8, 256, 44032, 2048), (16, 256, 1024, 4096), (16, 256, 32768, 4096), (32, 256, 11264, 8192)]
APART = [(32, 128, 1024, 4096), (36, 128, 1024, 4608), (40, 128, 5632, 5120), (48, 128, 5632, 6144), (64, 128, 1024, 8192), (64, 128, 5632, 8192), (64, 64, 5632, 4096), (32, 128, 16384, 4096),
         (32, 128, 32768, 4096), (64, 64, 22016, 4096), (40, 128, 32768, 5120), (48, 128, 32768, 6144), (56, 128, 22016, 7168), (64, 128, 14336, 8192), (64, 128, 44032, 8192),
         (32, 256, 32768, 8192), (96, 64, 22016, 4096)]


@pytest.mark.parametrize("case", TOGETHER + APART)
def test_gate_up_beside_the_delta_step(case):
    assert _delta(*case) == (case in TOGETHER)


@pytest.mark.parametrize("dim", [64, 128, 256])
def test_never_what_the_launch_cannot_take(dim):
    assert not _delta(16, dim, 1024, 1024, torch.float32) and not _delta(16, dim, 8192, 8256) and not _delta(16, dim, 1024, 1028)


def _moe(slots, ff, K, out_k, dt=torch.bfloat16):
    from llava_mi355x import _C
    f = ctypes.c_int32()
    _C.check(_C.lib.lmx_op_moe_joins(_C.torch_dtype_code(dt), slots, ff, K, out_k, f))
    return bool(f.value)


# experts of a row, their width, the layer's width, the output projection's columns
BESIDE = [(4, 704, 1024, 1024), (4, 1408, 2048, 2048), (4, 4096, 2048, 2048), (8, 4096, 2048, 2048), (4, 4096, 3072, 3072), (8, 4096, 3072, 3072), (4, 256, 4096, 4096), (4, 1408, 4096, 4096),
          (4, 2752, 3584, 3584), (4, 2752, 4096, 4096), (4, 3328, 4096, 4096), (2, 2048, 4096, 4096), (2, 5632, 4096, 4096), (8, 1408, 4096, 4096), (8, 704, 3584, 3584)]
ALONE = [(4, 4096, 4096, 4096), (4, 8192, 4096, 4096), (2, 4096, 4096, 4096), (8, 2048, 3584, 3584), (8, 2048, 4096, 4096), (8, 4096, 4096, 4096), (4, 4096, 3584, 3584), (8, 5632, 4096, 4096),
         (4, 4096, 5120, 4096), (4, 2048, 6144, 4096), (4, 4096, 6144, 4096), (4, 2048, 7168, 4096), (4, 4096, 8192, 4096)]


@pytest.mark.parametrize("case", BESIDE + ALONE)
def test_output_projection_beside_the_experts(case):
    assert _moe(*case) == (case in BESIDE)


def test_never_more_columns_than_the_launch_stages():
    assert not _moe(4, 1408, 2048, 4160) and not _moe(4, 1408, 2048, 2048, torch.float32) and not _moe(4, 1408, 2048, 2052)
