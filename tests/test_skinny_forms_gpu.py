"""Linears of a decode batch over every form the cost rule picks (csrc/skinny.hip: skinny_form): 1, 2 and 4 row tiles, 1, 2 and 4 K slices, row counts at the token tiles' edges, N with
a remainder of 8 and of 16 rows, K of one super-step, of an odd number and (plain loads) of a part of one.  Against float64 within the bound of an fp32 sum rounded once to
16 bits; the fragment-order copy (21, the engine's) and the layout as it is (20) give the same bits, K slices (24) the same sums in another order, and again the same
bits on scratch and tickets that another input has used."""
import pytest
import torch

pytestmark = pytest.mark.gpu
# N, K: (row tiles, K slices) of up to 8, up to 16 and more rows
SHAPES = {(8, 128): [(1, 1)] * 3, (1048, 384): [(1, 1)] * 3, (1040, 160): [(1, 1)] * 3, (2048, 5632): [(1, 1)] * 3, (4096, 4096): [(1, 1)] * 3, (4096, 11008): [(1, 1), (1, 1), (2, 2)],
          (5120, 13824): [(2, 1), (2, 1), (4, 2)], (6208, 2048): [(2, 1)] * 3, (12288, 1152): [(1, 1), (4, 1), (4, 1)], (640, 13824): [(1, 4)] * 3, (1088, 11008): [(1, 2)] * 3,
          (2048, 13824): [(1, 2), (1, 2), (2, 4)], (4032, 13824): [(1, 1), (1, 1), (4, 4)], (8192, 1024): [(1, 1), (2, 1), (2, 1)]}


def test_every_form_is_here():
    """What the rule picks over all widths of whole 64s below 8192 and some above, and what it picks for the shapes of this file."""
    from llava_mi355x import ops
    form = lambda M, N, K: ops.gemm_form(torch.bfloat16, M, N, K, batch=True)[1:]
    picked = {form(M, N, K) for M in (1, 8, 9, 16, 17, 32) for N in list(range(64, 8192, 64)) + [8200, 12288, 15360, 22016, 32000] for K in (128, 512, 2048, 4096, 5632, 11008, 13824)}
    assert picked == {form(M, N, K) for M in (1, 15, 16, 17, 32) for N, K in SHAPES}
    for (N, K), want in SHAPES.items():
        for M, i in ((1, 0), (8, 0), (9, 1), (16, 1), (17, 2), (32, 2)):
            assert form(M, N, K)[::2] == want[i], (M, N, K)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K", list(SHAPES))
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
    ops.gemm(2 - x, w, variant=24)
    assert torch.equal(sliced, ops.gemm(x, w, variant=24))
