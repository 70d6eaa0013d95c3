"""SiLU and quick GELU over the whole range of their exponential (csrc/common.h: act_silu, act_quick_gelu): results down to 2^-120, where the denominator is 2^126 and more, against
float64.  The argument reaches the epilogue exactly (one weight of 1 a row, zeros).  Tolerance: the result's rounding (half a unit in the last place: 2^-8, 2^-24), and the exponential's,
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


def _sums(dt, act, M):
    """act of sums of two operands, exact in 32 bits, 1024 a row: the results and the arguments"""
    from llava_mi355x import ops
    g = torch.Generator(device="cuda").manual_seed(act + M)
    z = (4 * torch.randn(M, 1, generator=g, device="cuda")).clamp(-15, 15).mul(16).round().div(16).to(dt)          # eight bits, and six more behind them: their sum has no more than 15
    lo = (torch.randint(-63, 64, (1024,), generator=g, device="cuda") / 2048).to(dt)
    x = torch.zeros(M, 1024, device="cuda", dtype=dt)
    x[:, :1], x[:, 1] = z, 1.0
    gate = torch.zeros(1024, 1024, device="cuda", dtype=dt)
    gate[:, 0], gate[:, 1] = 1.0, lo
    w = gate
    if act == 3:
        w = torch.zeros(2048, 1024, device="cuda", dtype=dt)
        w.view(32, 2, 32, 1024)[:, 0] = gate.view(32, 32, 1024)
        w.view(32, 2, 32, 1024)[:, 1, :, 1] = 1.0
    return ops.gemm(x, w, act=act, out=torch.empty(M, 1024, device="cuda", dtype=dt)), z.double() + lo.double()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("act", [1, 3])
@pytest.mark.parametrize("M", [1, 12, 139, 300, 1200])
def test_a_result_is_rounded_once(cuda, dt, act, M):
    """The result's own rounding, at the exact half unit, and what 32 bits add: the exponential's and the quotient's, 4 units of 2^-23 (3.9 over all arguments; an exponent rounded to 32 bits
    adds |cx| / 2, 16 here)."""
    got, a = _sums(dt, act, M)
    got = got.double()
    ref = a / (1 + torch.exp(-a * (float(torch.tensor(1.702)) if act == 1 else 1.0)))
    bits = {torch.bfloat16: 8, torch.float16: 11, torch.float32: 24}[dt]
    exponent = torch.frexp(ref).exponent.double()
    half = torch.exp2(torch.maximum(exponent, torch.full_like(exponent, -13.0)) - bits - 1) if dt == torch.float16 else torch.exp2(exponent - bits - 1)
    err = (got - ref).abs() - half
    assert (err <= 4 * 2.0 ** -23 * ref.abs()).all(), float((err / ref.abs().clamp_min(1e-30)).max() * 2 ** 23)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", [1, 3])
@pytest.mark.parametrize("M", [12, 139, 300, 1200])
def test_sixteen_bits_are_the_rounded_thirty_two(cuda, dt, act, M):
    """The quotient of 16-bit outputs is the division's but for the last of 32 bits in a hundredth of the arguments, so no more than one result in 2^16 is rounded the other way than the fp32
    model's (a hundredth of 2^-13, the share of a half unit that one such bit is, and 8 times that; half of the quotients off by a bit would be one in 2^14)."""
    got, want = _sums(dt, act, M)[0], _sums(torch.float32, act, M)[0].to(dt)
    assert int((got != want).sum()) <= got.numel() / 65536
