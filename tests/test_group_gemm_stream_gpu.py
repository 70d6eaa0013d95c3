"""Grouped products on tiles of 32 and 64 rows (csrc/moe.hip: group_gemm_kernel): plain loads, weights marked streaming with every
tile's walk over K begun somewhere else, and two slabs (group_gemm_form: from 224 and from 513 to 1024 workgroups with work), on both sides of each line."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16}


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("bm,rows,per_row,E,N", [(32, 32, 4, 16, 3264), (32, 32, 4, 16, 3328), (32, 96, 4, 16, 2560), (32, 97, 4, 16, 2560), (32, 104, 4, 16, 264), (64, 204, 4, 16, 264),
                                                 (64, 205, 4, 16, 264), (32, 5, 3, 15, 4480), (32, 16, 1, 16, 4096), (32, 24, 4, 16, 1664), (32, 24, 4, 16, 1792), (32, 32, 4, 16, 4096),
                                                 (32, 32, 4, 16, 4104), (32, 12, 4, 16, 8192), (32, 12, 4, 16, 8200), (64, 80, 4, 16, 1664), (64, 80, 4, 16, 1792)])
@pytest.mark.parametrize("K", [64, 128, 192, 704])
def test_products(cuda, dt, bm, rows, per_row, E, N, K):
    from llava_mi355x import ops
    g = torch.Generator(device="cuda").manual_seed(rows + N + K)
    x = torch.randn(rows, K, generator=g, device="cuda").to(DT[dt])
    w = (torch.randn(E, N, K, generator=g, device="cuda") / K ** 0.5).to(DT[dt])
    ids = torch.randint(0, E, (rows, per_row), generator=g, device="cuda", dtype=torch.int32)
    got = ops.group_gemm(x, w, ids, bm=bm).view(rows, per_row, N)
    wd = w.double()
    for j in range(per_row):
        want = torch.empty(rows, N, dtype=torch.float64, device="cuda")
        for e in range(E):
            at = ids[:, j] == e
            want[at] = x[at].double() @ wd[e].t()
        err = (got[:, j].double() - want).abs()
        ulp = 2.0 ** (-8 if dt == "bf16" else -11) * want.abs() + 2e-5 * float(want.abs().max()) + (2.0 ** -25 if dt == "f16" else 0)      # half a unit of the result, and the 32-bit sums
        assert bool((err <= ulp).all()), float((err / ulp).max())
    assert torch.equal(got, ops.group_gemm(x, w, ids, bm=bm).view(rows, per_row, N))
