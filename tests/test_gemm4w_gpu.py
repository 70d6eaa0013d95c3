"""The four-wave GEMM (csrc/gemm4w.h, variants 100 mb + 10 nb + slices of lmx_op_gemm): every tile form at the edges of its tiles and of its ring, against the float64 product rounded
once (one unit in the last place, as tests/test_gemm8p_gpu.py), and the choice between the forms."""
import math

import pytest
import torch

from test_gemm8p_gpu import DT, _mk, assert_one_ulp

FORMS = [88, 78, 77, 86, 58, 66, 56, 54, 45, 44]


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("form", FORMS)
def test_forms(cuda, dt, form):
    """One K-step; fewer K-steps than the ring holds, odd and even; a last row tile with and without rows in its second half; a last column tile of 4, 8 and more columns; one full tile."""
    from llava_mi355x import ops
    BM, BN = 32 * (form // 10), 32 * (form % 10)
    for M, N, K in [(BM, BN, 64), (BM + 1, BN + 4, 128), (3, 8, 192), (BM // 2, 2 * BN - 12, 256), (2 * BM - 15, BN + 24, 320), (BM + BM // 2 + 1, 136, 576), (1087, 3 * BN + 40, 1024)]:
        x, w = _mk(M, N, K, dt, cuda, M * 7 + N + K)
        ref = x.double() @ w.double().t()
        one = ops.gemm(x, w, variant=10 * form + 1)
        assert_one_ulp(one, ref, dt, 2e-5 * float(ref.abs().max()), f"form {form} {M}x{N}x{K}")
        if N % 8 == 0:                                                       # the same products in the same order, whatever the tile: the same bits
            assert torch.equal(one, ops.gemm(x, w, variant=35))
        for S in (2, 3):
            got = ops.gemm(x, w, variant=10 * form + S)
            assert_one_ulp(got, ref, dt, 2e-5 * float(ref.abs().max()), f"form {form} {M}x{N}x{K}, {S} slices")


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("act", [0, 1, 2])
def test_epilogues(cuda, form, act):
    from llava_mi355x import ops
    M, N, K = 700, 520, 640
    x, w = _mk(M, N, K, "bf16", cuda, act + form)
    b = torch.randn(N, device=cuda).bfloat16(); r = torch.randn(M, N, device=cuda).bfloat16()
    y = x.double() @ w.double().t() + b.double()
    if act == 1:
        y = y * torch.sigmoid(1.702 * y)
    elif act == 2:
        y = torch.nn.functional.gelu(y)
    ref = y + r.double()
    for S in (1, 2):
        v = 10 * form + S
        got = ops.gemm(x, w, bias=b, residual=r, act=act, variant=v)
        assert_one_ulp(got, ref, "bf16", 3e-5 * float(ref.abs().max()), f"variant {v} act {act}")
        r2 = r.clone()                                                       # in place: C aliases R
        ops.gemm(x, w, bias=b, residual=r2, act=act, variant=v, out=r2)
        assert torch.equal(r2, got)
        wide = torch.zeros(M, N + 4, device=cuda, dtype=torch.bfloat16)      # rows of 8-byte alignment
        ops.gemm(x, w, bias=b, residual=r, act=act, variant=v, out=wide[:, :N])
        assert torch.equal(wide[:, :N], got) and not bool(wide[:, N:].any())


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("M", [1, 77, 290])
def test_gated(cuda, form, M):
    """Outputs of one 16-column block are 8 gate and 8 up rows of the weight, whose own groups are 32 and 32; widths that end inside a tile."""
    from llava_mi355x import _C, ops
    for I in (32, 352, 512):
        K = 256
        g_ = torch.Generator(device=cuda).manual_seed(I + M)
        x = torch.randn(M, K, device=cuda, generator=g_).bfloat16()
        g, u = ((torch.randn(I, K, device=cuda, generator=g_) / math.sqrt(K)).bfloat16() for _ in range(2))
        fused = ops.interleave_gate_up(g, u)
        ref = torch.nn.functional.silu(x.double() @ g.double().t()) * (x.double() @ u.double().t())
        for S in (1, 2):
            got = ops.gemm(x, fused, act=_C.ACT_SILU_MUL, variant=10 * form + S)
            assert_one_ulp(got, ref, "bf16", 3e-5 * float(ref.abs().max()), f"form {form} gated {M}x{I}, {S} slices")


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("act", [0, 1, 2, 3, 4])
def test_three_slices(cuda, form, act):
    """Seven K-steps in slices of 2, 2 and 3 (one, one and two pairs): bias, activations, gating with a bias, the residual; row and column tails.  Against the un-sliced tiles' bound."""
    from llava_mi355x import _C, ops
    M, N, K = 290, 448, 448
    x, w = _mk(M, N, K, "bf16", cuda, act + form)
    b = torch.randn(N, device=cuda).bfloat16()
    y = x.double() @ w.double().t() + b.double()
    v = 10 * form + 3
    if act >= 3:
        y = y.view(M, N // 64, 2, 32)
        ref = ((torch.nn.functional.silu(y[:, :, 0]) if act == _C.ACT_SILU_MUL else torch.relu(y[:, :, 0])) * y[:, :, 1]).reshape(M, N // 2)
        got = ops.gemm(x, w, bias=b, act=act, variant=v, out=torch.empty(M, N // 2, device=cuda, dtype=torch.bfloat16))
        assert_one_ulp(got, ref, "bf16", 6e-5 * float(ref.abs().max()), f"variant {v} act {act}")
        return
    y = y * torch.sigmoid(1.702 * y) if act == 1 else torch.nn.functional.gelu(y) if act == 2 else y
    r = torch.randn(M, N, device=cuda).bfloat16()
    ref = y + r.double()
    got = ops.gemm(x, w, bias=b, residual=r, act=act, variant=v)
    assert_one_ulp(got, ref, "bf16", 3e-5 * float(ref.abs().max()), f"variant {v} act {act}")
    ops.gemm(x, w, bias=b, residual=r, act=act, variant=v, out=r)        # in place
    assert torch.equal(r, got)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,act", [(257, 10304, 1024, 0), (513, 4672, 640, 1), (700, 3072, 1024, 0), (1087, 4096, 4096, 0), (1087, 22016, 1024, 3), (2048, 2048, 5632, 0), (2679, 6400, 2048, 0), (6528, 4096, 1088, 0),
                                       (2693, 2048, 128, 0), (1348, 21056, 448, 3), (1200, 4096, 1024, 1), (1348, 21056, 1024, 3)])
def test_choice(cuda, M, N, K, act):
    """What variant 0 and a prefill's call take past the rule's line, the four-wave tiles and the forms that are cheaper there."""
    from llava_mi355x import _C, ops
    form = ops.gemm_form(torch.bfloat16, M, N, K, act=act)[0]
    assert form == {(700, 1024): 1, (2693, 128): 0, (1348, 448): 0, (1200, 1024): 1}.get((M, K), 2)
    x, w = _mk(M, N, K, "bf16", cuda, M + N)
    y = x.double() @ w.double().t()
    if act == 3:
        c = torch.arange(N // 2, device=cuda)
        rows = (c // 32) * 64 + c % 32
        y = torch.nn.functional.silu(y[:, rows]) * y[:, rows + 32]
    elif act == 1:
        y = y * torch.sigmoid(1.702 * y)
    for v in (0, _C.GEMM_SCRATCH):
        assert_one_ulp(ops.gemm(x, w, act=act, variant=v), y, "bf16", 3e-5 * float(y.abs().max()), f"{M}x{N}x{K} variant {v}")


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(513, 4672, 640), (1087, 4096, 4096), (2048, 5120, 1024)])
@pytest.mark.parametrize("odd", [1, 2, 3])
def test_residual_rows_of_any_pitch(cuda, dt, M, N, K, odd):
    """A residual whose rows are not multiples of 8 bytes apart, on the large side of the rule's lines: taken by another kernel, not refused."""
    from llava_mi355x import _C
    x, w = _mk(M, N, K, dt, cuda, M + odd)
    r = torch.randn(M, N + odd, device=cuda).to(DT[dt])
    ref = x.double() @ w.double().t() + r[:, :N].double()
    out = torch.empty(M, N, device=cuda, dtype=DT[dt])
    for v in (0, _C.GEMM_SCRATCH):
        _C.check(_C.lib.lmx_op_gemm(_C.torch_dtype_code(DT[dt]), _C.ptr(x), _C.ptr(w), _C.ptr(out), None, _C.ptr(r), M, N, K, K, K, N, N + odd, 0, v, _C.stream_handle()), "gemm")
        assert_one_ulp(out, ref, dt, 2e-5 * float(ref.abs().max()), f"{M}x{N}x{K} pitch {N + odd} variant {v}")


@pytest.mark.gpu
def test_refusals(cuda):
    from llava_mi355x import ops
    from llava_mi355x._C import LmxError
    x, w = _mk(300, 256, 128, "bf16", cuda, 1)
    for v in (331, 491, 701, 100):                                           # no such tiles
        with pytest.raises(LmxError):
            ops.gemm(x, w, variant=v)
    with pytest.raises(LmxError):
        ops.gemm(x[:, :96].contiguous(), w[:, :96].contiguous(), variant=881)                    # K % 64
