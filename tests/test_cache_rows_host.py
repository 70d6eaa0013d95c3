"""Memory that a row of the K / V^T caches takes (csrc/engine.h: kv_row_pitch), asked of the library on the host."""
import pytest
import torch


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
def test_cache_rows_take_at_most_a_sixteenth_more(dtype):
    """Capacities of 1 .. 16384 positions: what a cache row takes memory for, and that the decode kernels' 128-key chunks stay inside it."""
    from llava_mi355x import _C
    code = _C.torch_dtype_code(getattr(torch, dtype))
    for cap in list(range(1, 400)) + list(range(512, 16385, 64)):
        rows = -(-cap // 128) * 128
        pitch = _C.lib.lmx_kv_row_pitch(code, cap)
        assert pitch % 128 == 0 and rows <= pitch <= (rows if dtype == "float32" else rows + rows // 16), cap
        assert rows < 2048 or dtype == "float32" or pitch % 256 == 128, cap
    assert _C.lib.lmx_kv_row_pitch(code, 0) == _C.lib.lmx_kv_row_pitch(code, 2048)
