"""Linears of a few dozen to a few hundred rows (csrc/gemm_rows.hip): every form at the edges of its tiles — rows around 32 and 256, weight rows that fill no tile, fewer slabs of K
than the ring holds, slices of unequal length — against the float64 product rounded once (one unit in the last place, as tests/test_gemm8p_gpu.py derives it), and the rule
that sends a product here."""
import pytest
import torch

from test_gemm8p_gpu import DT, _mk, assert_one_ulp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("variant", [1101, 1103, 1201, 1202, 2101, 2202, 3203])
@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (31, 72, 192), (33, 136, 320), (128, 200, 448), (200, 776, 1024), (256, 128, 640), (257, 384, 1152), (500, 520, 704), (600, 264, 2048)])
def test_forms(cuda, dt, variant, M, N, K):
    from llava_mi355x import ops
    if -(-M // (variant // 1000)) > 256 or variant % 100 > K // 64:
        pytest.skip("not a form of this shape")
    x, w = _mk(M, N, K, dt, cuda, M + N + K + variant)
    ref = x.double() @ w.double().t()
    got = ops.gemm(x, w, variant=variant)
    assert_one_ulp(got, ref, dt, 2e-5 * float(ref.abs().max()), f"variant {variant} {M}x{N}x{K}")
    assert torch.equal(got, ops.gemm(x, w, variant=variant))


@pytest.mark.parametrize("variant", [1101, 1102, 1201, 1204, 2202])
@pytest.mark.parametrize("act", [0, 1, 2, 3, 4])
def test_epilogues(cuda, variant, act):
    from llava_mi355x import ops
    M, N, K = 139, 448, 832
    x, w = _mk(M, N, K, "bf16", cuda, act + variant)
    b = torch.randn(N, device=cuda).bfloat16()
    y = x.double() @ w.double().t() + b.double()
    if act >= 3:
        y = y.view(M, N // 64, 2, 32)
        ref = ((torch.nn.functional.silu(y[:, :, 0]) if act == 3 else torch.relu(y[:, :, 0])) * y[:, :, 1]).reshape(M, N // 2)
        got = ops.gemm(x, w, bias=b, act=act, variant=variant, out=torch.empty(M, N // 2, device=cuda, dtype=DT["bf16"]))
        assert_one_ulp(got, ref, "bf16", 6e-5 * float(ref.abs().max()), f"variant {variant} act {act}")
        return
    y = y * torch.sigmoid(1.702 * y) if act == 1 else torch.nn.functional.gelu(y) if act == 2 else y
    r = torch.randn(M, N, device=cuda).bfloat16()
    got = ops.gemm(x, w, bias=b, residual=r, act=act, variant=variant)
    assert_one_ulp(got, y + r.double(), "bf16", 3e-5 * float((y + r.double()).abs().max()), f"variant {variant} act {act}")
    ops.gemm(x, w, bias=b, residual=r, act=act, variant=variant, out=r)              # in place
    assert torch.equal(r, got)


@pytest.mark.parametrize("M,N,K,res", [(385, 2048, 2048, False), (577, 4096, 1024, False), (640, 2112, 4096, True), (1087, 4096, 4096, True), (1087, 4096, 4160, True), (2308, 1024, 1024, True),
                                       (2679, 1280, 2048, False), (4616, 1024, 1024, False), (1153, 1024, 2048, True), (600, 4096, 4096, True), (2308, 1024, 4096, False), (1200, 2048, 2048, True),
                                       (257, 6208, 2048, False)])
def test_one_round_of_tiles(cuda, M, N, K, res):
    """The other part of the rule: row tiles of a height that makes one round of workgroups, and both sides of its lines: small tiles below, four-wave tiles past 640 tiles of 64 x 64."""
    from llava_mi355x import ops
    form = ops.gemm_form(torch.bfloat16, M, N, K, scratch_bytes=0)
    assert form[0] == {(385, 2048): 0, (1153, 1024): 0, (1087, 4096): 2, (2679, 1280): 2, (4616, 1024): 2}.get((M, N), 1) and (form[0] != 1 or form[1] > 1)
    x, w = _mk(M, N, K, "bf16", cuda, M + N)
    r = torch.randn(M, N, device=cuda).bfloat16() if res else None
    ref = x.double() @ w.double().t() + (r.double() if res else 0)
    assert_one_ulp(ops.gemm(x, w, residual=r), ref, "bf16", 2e-5 * float(ref.abs().max()), f"{M}x{N}x{K}")


@pytest.mark.parametrize("M", [2, 32, 128, 129, 256, 257, 384, 385, 512, 513])
@pytest.mark.parametrize("N,K,ldc", [(12288, 1024, 12288), (22016, 1024, 22016), (12288, 1024, 12292), (4096, 4096, 4096)])
def test_rule(cuda, M, N, K, ldc):
    """What variant 0 takes, on both sides of every line of the rule (past 256 rows: of the width that the four-wave tiles leave to it) and with rows that are not 16-byte aligned
    (another kernel's)."""
    from llava_mi355x import ops
    x, w = _mk(M, N, K, "bf16", cuda, M)
    out = torch.zeros(M, ldc, device=cuda, dtype=DT["bf16"])
    got = ops.gemm(x, w, out=out[:, :N])
    ref = x.double() @ w.double().t()
    assert_one_ulp(got, ref, "bf16", 2e-5 * float(ref.abs().max()), f"{M}x{N}x{K}")
    assert ldc == N or not bool(out[:, N:].any())


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("form,M,N,K", [((1, 64, 2), 64, 6144, 3072), ((1, 64, 3), 33, 3072, 2048), ((1, 64, 4), 2, 2048, 3072), ((1, 128, 2), 129, 12288, 3072), ((1, 128, 4), 129, 8192, 8192),
                                        ((1, 128, 5), 200, 6144, 8192), ((1, 128, 6), 139, 3072, 8192), ((2, 128, 2), 257, 6144, 3072), ((2, 128, 3), 290, 5120, 3072), ((2, 128, 4), 257, 4096, 4096)])
def test_slices_of_the_rule(cuda, dt, form, M, N, K):
    """The slice counts that the rule itself picks with a prefill's scratch; three launches on the same slabs, another input between."""
    from llava_mi355x import _C, ops
    assert ops.gemm_form(DT[dt], M, N, K) == (1,) + form
    x, w = _mk(M, N, K, dt, cuda, M + N)
    r = torch.randn(M, N, device=cuda).to(DT[dt])
    ref = x.double() @ w.double().t() + r.double()
    got = ops.gemm(x, w, residual=r, variant=_C.GEMM_SCRATCH)
    assert_one_ulp(got, ref, dt, 2e-5 * float(ref.abs().max()), f"{M}x{N}x{K}")
    ops.gemm(-x, w, residual=r, variant=_C.GEMM_SCRATCH)
    assert torch.equal(got, ops.gemm(x, w, residual=r, variant=_C.GEMM_SCRATCH))


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(5, 10248, 1024), (139, 32000, 1024), (300, 8200, 2048)])
@pytest.mark.parametrize("cap", [0.0, 7.5])
def test_fp32_output_with_a_soft_cap(cuda, dt, M, N, K, cap):
    """An output head's logits.  Bound: an fp32 sum of K products (the cap's slope is at most 1), tanh and its division to 8 units in the last place."""
    from llava_mi355x import ops
    x, w = _mk(M, N, K, dt, cuda, M + N)
    w = w * 4
    want = x.double() @ w.double().t()
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    if cap:
        want = cap * torch.tanh(want / cap)
    got = ops.linear_f32(x, w, cap, 0)
    assert got.dtype == torch.float32 and bool(((got.double() - want).abs() <= bound + want.abs() * 2.0 ** -20).all())
