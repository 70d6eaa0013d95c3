"""The order in which a decode batch launches its sequences (csrc/attention.hip: batch_attn_order), asked of the library on the host."""
import ctypes
import random

import pytest


def _order(lens, heads):
    from llava_mi355x import _C
    n = len(lens)
    out = (ctypes.c_uint8 * n)()
    _C.check(_C.lib.lmx_op_batch_attn_order((ctypes.c_int32 * n)(*lens), n, heads, out))
    return list(out)


@pytest.mark.parametrize("heads", [1, 3, 32, 40, 64, 300])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 13, 16, 17, 32, 255, 256])
def test_every_sequence_once_and_long_ones_meet_short_ones(n, heads):
    lens = [random.Random(n * heads + i).randrange(1, 3000) for i in range(n)]
    order = _order(lens, heads)
    assert sorted(order) == list(range(n))
    half = -(-256 // heads)
    by = [lens[i] for i in order]
    first, second, rest = by[:half], by[half:2 * half], by[2 * half:]
    assert first == sorted(first, reverse=True) and second == sorted(second) and rest == sorted(rest, reverse=True)
    assert not second or (min(first) >= max(second) and (not rest or min(second) >= max(rest)))


def test_equal_lengths_stay_in_place_and_bad_arguments_raise():
    from llava_mi355x import _C
    assert _order([5] * 8, 32) == list(range(8))
    for n, heads in [(0, 32), (257, 32), (4, 0)]:
        with pytest.raises(_C.LmxError):
            _C.check(_C.lib.lmx_op_batch_attn_order((ctypes.c_int32 * 257)(), n, heads, (ctypes.c_uint8 * 257)()))


@pytest.mark.parametrize("n,heads,want", [(12, 40, True), (13, 40, False), (14, 40, False), (15, 40, True), (25, 20, True), (26, 20, False), (27, 20, True), (16, 32, True), (17, 32, True), (16, 31, True),
                                          (17, 31, False), (18, 31, False), (19, 31, True), (1, 600, False), (3, 300, True), (256, 1, True), (256, 256, True)])
def test_no_long_one_last(n, heads, want):
    """The reversed ones end within the first 512 workgroups, or others follow them."""
    from llava_mi355x import _C
    f = ctypes.c_int32()
    _C.check(_C.lib.lmx_op_batch_attn_ordered(n, heads, f))
    assert bool(f.value) == want
