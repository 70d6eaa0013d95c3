"""Grouped products of mixtures (csrc/moe.hip, the grouped form of csrc/gemm4w.h): every tile form against the float64 product rounded once (one unit in the last place, as
tests/test_gemm8p_gpu.py) and, gated, against the group's rows through the same tiles of lmx_op_gemm: the same bits."""
import pytest
import torch

from test_gemm8p_gpu import DT, assert_one_ulp

FORMS = [(8, 8), (7, 8), (7, 7), (8, 6), (5, 8), (6, 6), (5, 6), (5, 4), (4, 5), (4, 4)]


def mixture(cuda, dt, rows, top, E, N, K, shared, seed):
    """x, w, ids: expert 1 is nobody's choice, expert 0 everybody's; the others get what is left at random"""
    g = torch.Generator(device=cuda).manual_seed(seed)
    x = torch.randn(rows if shared else rows * top, K, device=cuda, generator=g).to(DT[dt])
    w = (torch.randn(E, N, K, device=cuda, generator=g) * K ** -0.5).to(DT[dt])
    rest = 2 + torch.rand(rows, E - 2, device=cuda, generator=g).argsort(1)[:, :top - 1]
    return x, w, torch.cat([torch.zeros_like(rest[:, :1]), rest], 1).int().contiguous()


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("form", [(1, 0), (2, 0), (0, 0)] + FORMS)
def test_forms(cuda, dt, form):
    """One K-step, odd and even counts of them; last row tiles with and without rows in their second half; column tails of 4 and 8; tiles with one row; an empty group."""
    from llava_mi355x import _C, ops
    mb, nb = form
    for rows, top, E, N, K, shared in [(1, 2, 4, 64, 64, True), (32 * mb + 1, 2, 5, 32 * nb + 12, 192, True), (300, 3, 6, 320, 320, True), (257, 2, 4, 200, 128, False), (700, 4, 16, 448, 576, True)]:
        x, w, ids = mixture(cuda, dt, rows, top, E, N, K, shared, rows + N)
        xs = x.repeat_interleave(top, 0) if shared else x
        got = ops.group_gemm(x, w, ids, shared_x=shared, bm=32 * mb, nb=nb)
        ref = torch.empty(rows * top, N, dtype=torch.float64, device=cuda)
        for e in range(E):
            at = (ids.reshape(-1) == e).nonzero()[:, 0]
            ref[at] = xs[at].double() @ w[e].double().t()
        assert_one_ulp(got, ref, dt, 2e-5 * float(ref.abs().max()), f"form {form} {rows} x {top}, {N} x {K}")
        if N % 64 or nb == 0:
            continue
        for act in (_C.ACT_SILU_MUL, _C.ACT_RELU_MUL):
            gated = ops.group_gemm(x, w, ids, act=act, shared_x=shared, bm=32 * mb, nb=nb)
            for e in range(E):
                at = (ids.reshape(-1) == e).nonzero()[:, 0]
                one = torch.empty(len(at), N // 2, dtype=x.dtype, device=cuda)
                if len(at):
                    assert torch.equal(gated[at], ops.gemm(xs[at].contiguous(), w[e], act=act, variant=100 * mb + 10 * nb + 1, out=one)), (form, rows, e)
