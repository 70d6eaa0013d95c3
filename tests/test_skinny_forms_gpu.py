"""Linears of a decode batch over every form the cost rule picks (csrc/skinny.hip: skinny_form): 1, 2 and 4 row tiles, 1, 2 and 4 K slices, row counts at the token tiles' edges, N with
a remainder of 8 and of 16 rows, K of one super-step, of an odd number and (plain loads) of a part of one.  Against float64 within the bound of an fp32 sum rounded once to
16 bits; the fragment-order copy (21, the engine's) and the layout as it is (20) give the same bits, K slices (24) the same sums in another order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(8, 128), (1048, 384), (1040, 160), (2048, 5632), (4096, 4096), (4096, 11008), (5120, 13824), (6208, 2048), (12288, 1152)])
def test_forms(cuda, dt, M, N, K):
    from llava_mi355x import ops
    g = torch.Generator(device=cuda).manual_seed(M + N + K)
    x = torch.randn(M, K, device=cuda, generator=g).to(dt); w = (torch.randn(N, K, device=cuda, generator=g) / K ** 0.5).to(dt)
    want = x.double() @ w.double().t()
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + want.abs() * (2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11) + 1e-7
    plain, copy, sliced = (ops.gemm(x, w, variant=v) for v in (20, 21, 24))
    assert torch.equal(plain, copy)
    for got in (copy, sliced):
        assert bool(((got.double() - want).abs() <= bound).all())
