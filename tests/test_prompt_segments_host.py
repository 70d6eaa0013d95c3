"""Workgroups of the launches over the rows of several sequences (csrc/kernels.h: row_segs_at, csrc/attention.hip: flash_segs_plan) and the scratch of their latent layers
(csrc/stack_mixers.cpp: latent_prefill_scratch), asked of the library on the host."""
import ctypes

import pytest


def plan(lens, heads, D=128, pos0=None, window=0):
    from llava_mi355x import ops
    return ops.flash_segs_plan(lens, pos0 or [0] * len(lens), heads, D, window)


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


@pytest.mark.parametrize("lens,pos0,heads,window,rows", [
    ([2048, 2048], None, 32, 0, 128), ([30] * 31 + [4096], None, 32, 0, 128), ([128, 128], [700, 640], 256, 0, 128), ([2048, 2048], None, 32, 1024, 128),      # the chip full of whole blocks
    ([900] * 4, None, 32, 0, 64), ([64] * 32, None, 32, 0, 64), ([129, 129], [900, 900], 256, 0, 64),                                                          # full, but of rows that are none
    ([1100, 894, 688], None, 16, 0, 64), ([128, 128], [700, 100], 140, 0, 64), ([2048, 30], None, 15, 0, 64),                                                   # CUs without work, blocks of unlike length
])
def test_larger_blocks_where_they_fill_the_chip(lens, pos0, heads, window, rows):
    assert plan(lens, heads, 128, pos0, window)[0] == rows


def test_the_narrow_heads_have_one_form():
    assert plan([1], 1, 64)[0] == plan([2048, 2048], 32, 64)[0] == 128


@pytest.mark.parametrize("lens,heads,D", [([], 4, 128), ([1] * 33, 4, 128), ([0], 4, 128), ([5], 0, 128), ([5], 4, 256)])
def test_bad_arguments_raise(lens, heads, D):
    from llava_mi355x import _C
    n = len(lens)
    with pytest.raises(_C.LmxError):
        _C.check(_C.lib.lmx_op_flash_segs_plan(D, heads, 0, n, (ctypes.c_int32 * 33)(*lens), (ctypes.c_int32 * 33)(), (ctypes.c_int32 * 2)(), None, 0))


@pytest.mark.parametrize("width,latent,window", [(4096, 512, 0), (2048, 256, 1024)])
def test_latent_scratch_of_many_rows(width, latent, window):
    """Queries and latents of all rows; keys and values, by row and in caches, of 8192 rows or of the longest prompt."""
    from llava_mi355x import _C
    size = lambda rows, keys, n: _C.lib.lmx_op_latent_scratch_bytes(_C.DTYPE_BF16, width, latent, window, rows, keys, n)  # noqa: E731
    row = lambda w: w * 2  # noqa: E731
    for prompts, n in ((2000, 32), (300, 200), (64, 32), (20000, 2)):
        rows, apart = prompts * n, max(8192, prompts)
        assert size(rows, prompts, n) <= rows * row(width + latent) + (2 * apart + 2 * (apart + 127 * 32)) * row(width) + 5 * 256
        assert size(rows, prompts, n) >= rows * row(width)
    assert size(2000, 2000, 1) <= 2000 * row(width) + (2 * 2000 + 2 * 2048) * row(width) + 5 * 256      # a prompt alone
    assert size(0, 1, 1) == size(1, 0, 1) == size(1, 1, 0) == 0

