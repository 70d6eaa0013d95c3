"""SiLU and quick GELU over the whole range of their exponential (csrc/common.h: over_one_plus_exp): results down to 2^-120, where the denominator is 2^126 and more, against
float64.  The argument reaches the epilogue exactly (one weight of 1 a row, zeros).  Tolerance: the result's rounding (half a unit in the last place: 2^-9, 2^-25), and the exponential's,
whose argument is rounded in 32 bits: (|cx| + 4) 2^-23.  Past the largest 32-bit exponential the result is 0, at most 2^-120 away."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("act", [1, 3])
@pytest.mark.parametrize("M", [1, 12, 300, 1200])
def test_the_whole_range(cuda, dt, act, M):
    from llava_mi355x import ops
    z = torch.linspace(-92.0, 92.0, 1200, dtype=torch.float64).to(dt).to(cuda)
    if act == 1:
        z = (z.double() / 1.702).to(dt)
    z = z[:: 1200 // M][:M] if M > 1 else z[25:26]
    x = torch.zeros(M, 1024, device=cuda, dtype=dt)
    x[:, 0], x[:, 1] = z, 1.0
    w = torch.zeros(2048, 1024, device=cuda, dtype=dt)
    w.view(32, 64, 1024)[:, :, 0] = 1.0
    if act == 3:
        w.view(32, 2, 32, 1024)[:, 1, :, 0], w.view(32, 2, 32, 1024)[:, 1, :, 1] = 0.0, 1.0
    out = torch.empty(M, 2048 // (2 if act == 3 else 1), device=cuda, dtype=dt)
    got = ops.gemm(x, w, act=act, out=out).double()
    zd = z.double()[:, None]
    cx = zd * (1.702 if act == 1 else 1.0)
    ref = (zd / (1 + torch.exp(-cx))).expand_as(got)
    tol = ref.abs() * ((2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -24) + (cx.abs() + 4) * 2.0 ** -23)
    tol = torch.where(cx < -88.7, torch.full_like(tol, 2.0 ** -120), tol)
    assert torch.isfinite(got).all() and ((got - ref).abs() <= tol).all(), ((got - ref).abs() / tol.clamp_min(1e-300)).max()
