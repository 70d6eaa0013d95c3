"""Which windowed decode kernel a step takes and how many splits (csrc/stack_ops.hip: decode_win_form), asked of the library on the host."""
import ctypes

import pytest
import torch


def _form(H, G, D, n, span, dt=torch.bfloat16):
    from llava_mi355x import _C
    f = (ctypes.c_int32 * 2)()
    _C.check(_C.lib.lmx_op_decode_win_form(_C.torch_dtype_code(dt), D, H, G, n, span, f))
    return bool(f[0]), f[1]


# heads, kv heads, width, sequences, keys: where one kernel measured at least a tenth faster than the other
GROUPED = [(32, 8, 128, 32, 1151), (32, 8, 128, 8, 130), (16, 4, 128, 4, 1200), (24, 12, 128, 2, 600), (8, 1, 128, 32, 600), (32, 32, 128, 8, 1200), (32, 32, 128, 2, 300), (16, 16, 64, 8, 130), (16, 1, 128, 32, 1200), (32, 8, 64, 2, 600)]
APART = [(32, 8, 128, 2, 20), (8, 1, 128, 2, 600), (8, 1, 128, 8, 60), (16, 1, 128, 4, 600), (32, 32, 128, 16, 60), (24, 12, 128, 32, 60), (16, 16, 64, 8, 60), (28, 4, 128, 2, 130)]


@pytest.mark.parametrize("case", GROUPED + APART)
def test_the_faster_kernel(case):
    assert _form(*case)[0] == (case in GROUPED)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G", [(32, 32), (24, 12), (32, 8), (16, 4), (8, 1), (17, 1), (40, 8)])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_splits(dt, H, G, D):
    """One round of workgroups for the grouped kernel, never more splits than chunks of 128 keys or than the scratch of a sequence holds, never a form that the kernel cannot take."""
    for n in (1, 2, 3, 5, 8, 13, 32, 200):
        for span in (1, 21, 127, 128, 129, 600, 1151, 4096, 100000):
            grouped, splits = _form(H, G, D, n, span, dt)
            assert 1 <= splits <= min(32, -(-span // 128))
            assert splits == 1 or (not grouped) or G * n * splits <= 256
            assert not grouped or (dt != torch.float32 and D <= 128 and H // G <= 16 and n > 1)


def _waves(H, G, D, n, max_len, window, dt=torch.bfloat16):
    from llava_mi355x import _C
    w = ctypes.c_int32()
    _C.check(_C.lib.lmx_op_decode_win_form_waves(_C.torch_dtype_code(dt), D, H, G, n, max_len, window, w))
    return w.value


# heads, kv heads, width, sequences, cached keys, window: steps timed with four and with eight waves a workgroup, all of them faster by more than the noise or level
EIGHT = [(32, 8, 128, 32, 1024, 1024), (32, 8, 128, 32, 513, 0), (32, 8, 128, 22, 1500, 0), (32, 8, 64, 32, 800, 0), (24, 12, 128, 16, 1100, 0), (32, 8, 128, 16, 1100, 0), (32, 8, 128, 11, 1500, 1024),
         (32, 8, 128, 16, 1900, 0), (16, 4, 128, 21, 3300, 0), (32, 8, 128, 8, 2150, 0), (16, 4, 128, 11, 2650, 0), (32, 4, 128, 32, 1250, 0)]
FOUR = [(32, 8, 128, 32, 512, 0), (32, 8, 128, 11, 1500, 0), (32, 8, 128, 16, 1524, 0), (16, 4, 128, 32, 1500, 0), (24, 12, 128, 8, 1500, 0), (24, 12, 128, 8, 1900, 0), (32, 32, 128, 8, 1500, 0),
        (32, 32, 128, 4, 1500, 0), (16, 4, 128, 21, 2150, 0), (32, 8, 128, 8, 2600, 0), (16, 4, 128, 11, 3300, 0), (32, 8, 128, 11, 600, 256), (32, 8, 128, 1, 1500, 0), (32, 8, 128, 33, 1500, 0),
        (32, 8, 256, 16, 1100, 0)]


@pytest.mark.parametrize("case", EIGHT + FOUR)
def test_waves_of_a_workgroup(case):
    assert _waves(*case) == (8 if case in EIGHT else 4) and _waves(*case, dt=torch.float32) == 4


@pytest.mark.parametrize("window,first", [(0, 1025), (1024, 1025), (1023, 1025), (963, 1025), (962, None), (700, None)])
def test_a_window_counts_by_the_pieces_it_can_touch(window, first):
    """16 sequences of 8 kv heads walk their keys in two splits: eight waves from the 17th piece of 64 keys on.  A window of w sees w - 1 cached keys, at most
    1 + ceil((w - 2) / 64) pieces."""
    assert [_waves(32, 8, 128, 16, n, window) for n in (1023, 1024)] == [4, 4]
    assert (_waves(32, 8, 128, 16, 1025, window) == 8) == (first == 1025)
