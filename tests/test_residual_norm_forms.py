"""The residual norm's two forms (csrc/stack_ops.hip: residual_norm_ahead): which one a launch takes, asked on the host, and that they are the same bits on both sides of every line."""
import ctypes

import pytest
import torch

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
# type, rows, width, injected row: rows that are one round without the loads ahead and two with them
PLAIN = [("bf16", 1537, 4096, 0), ("f16", 2048, 2112, 0), ("bf16", 769, 4160, 0), ("f16", 1536, 8192, 0), ("bf16", 1024, 8192, 1), ("bf16", 2560, 6144, 0), ("bf16", 1800, 3072, 1), ("f32", 1793, 2048, 0), ("f32", 1025, 4096, 1), ("f32", 513, 8192, 0)]
AHEAD = [("bf16", 1, 8192, 0), ("bf16", 2048, 2048, 0), ("f16", 1536, 4096, 0), ("bf16", 2049, 4096, 0), ("bf16", 1700, 4096, 1), ("f16", 768, 8192, 0), ("bf16", 1537, 8192, 1), ("bf16", 2561, 8192, 0), ("f32", 1792, 2048, 0),
         ("f32", 1024, 4096, 0), ("f32", 512, 8192, 1)]


@pytest.mark.parametrize("case", PLAIN + AHEAD)
def test_form(case):
    from llava_mi355x import _C
    f = ctypes.c_int32()
    _C.check(_C.lib.lmx_op_residual_norm_form(_C.torch_dtype_code(DT[case[0]]), *case[1:], f))
    assert bool(f.value) == (case in AHEAD)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,rows,H,inject", PLAIN)
def test_both_forms_are_the_same_bits(cuda, dt, rows, H, inject):
    """All rows in one launch, and the same rows a few at a time, where the loads run ahead."""
    from llava_mi355x import ops
    g = torch.Generator(device="cuda").manual_seed(rows + H)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y, inj, post, pre = r(rows, H), r(rows, H).to(DT[dt]), r(rows, H).to(DT[dt]), r(H).to(DT[dt]), r(H).to(DT[dt])
    one = ops.residual_norm(x, y, post, inj if inject else None, pre, 0.37, 1e-5, dtype=DT[dt])
    for a in range(0, rows, 200):
        few = ops.residual_norm(x[a:a + 200], y[a:a + 200], post, inj[a:a + 200] if inject else None, pre, 0.37, 1e-5, dtype=DT[dt])
        assert torch.equal(one[0][a:a + 200], few[0]) and torch.equal(one[1][a:a + 200], few[1])
