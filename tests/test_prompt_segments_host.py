"""Workgroups of the launches over the rows of several sequences (csrc/kernels.h: row_segs_at, csrc/attention.hip: flash_segs_plan), asked of the library on the host."""
import ctypes

import pytest


def plan(lens, heads, D=128, pos0=None):
    """(query rows of a workgroup, [(sequence, its workgroup)])"""
    from llava_mi355x import _C
    n, cap = len(lens), sum(-(-k // 64) for k in lens) * heads + 1
    form, out = (ctypes.c_int32 * 2)(), (ctypes.c_int32 * (2 * cap))()
    _C.check(_C.lib.lmx_op_flash_segs_plan(D, heads, n, (ctypes.c_int32 * n)(*lens), (ctypes.c_int32 * n)(*(pos0 or [0] * n)), form, out, cap))
    assert form[1] < cap
    return form[0], [(out[2 * b], out[2 * b + 1]) for b in range(form[1])]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("heads", [1, 3, 32])
@pytest.mark.parametrize("lens", [[1], [64], [65], [1, 1], [30] * 31 + [2000], [129, 70, 1, 200, 33], [128] * 32, list(range(1, 33)), [7, 4000]])
def test_every_block_of_every_sequence_once(lens, heads, D):
    rows, blocks = plan(lens, heads, D)
    assert sorted(blocks) == [(i, b) for i, n in enumerate(lens) for b in range(-(-n // rows) * heads)]


def test_most_keys_first():
    order = lambda lens, pos0=None: list(dict.fromkeys(s for s, _ in plan(lens, 2, pos0=pos0)[1]))  # noqa: E731
    assert order([30, 2000, 64]) == [1, 2, 0]
    assert order([30, 200, 64], [900, 0, 136]) == [0, 1, 2]      # 930, 200 and 200 keys: equal ones as they come


@pytest.mark.parametrize("lens,heads,D", [([], 4, 128), ([1] * 33, 4, 128), ([0], 4, 128), ([5], 0, 128), ([5], 4, 256)])
def test_bad_arguments_raise(lens, heads, D):
    from llava_mi355x import _C
    n = len(lens)
    with pytest.raises(_C.LmxError):
        _C.check(_C.lib.lmx_op_flash_segs_plan(D, heads, n, (ctypes.c_int32 * 33)(*lens), (ctypes.c_int32 * 33)(), (ctypes.c_int32 * 2)(), None, 0))
