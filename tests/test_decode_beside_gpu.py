"""One sequence's decode step: launches that two products share (csrc/delta.hip: delta_decode_linear_kernel, csrc/moe.hip: group_gemv_linear_kernel) against the launches of their own,
and the forms of the linear that forms its own row (csrc/gemm.hip: launch_gemv2_res) on both sides of their lines."""
import ctypes

import pytest
import torch

from oracle import vizosun_oracle as O
from vizosun_util import build_config, config, delta, dense, latent, moe, rel, steady_routing

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16}
TOL = {"bf16": 4e-2, "f16": 6e-3}


def _steps(m, first, n):
    """logits of n steps, one at a time, behind a prompt of 5 tokens"""
    from llava_mi355x._C import check, lib, ptr, stream_handle
    from llava_mi355x.engine_lm import LmxKVCache
    cache, out = LmxKVCache(m, 1), []
    e = m.get_model().embed_tokens(torch.tensor(first, device="cuda"))
    check(lib.lmx_prefill(m._h, cache.seqs[0], ptr(e), len(first), 0, None, 0, 1, stream_handle()), "lmx_prefill")
    for i in range(n):
        z = torch.empty((1, m._vocab_cap), dtype=m.logits_dtype, device="cuda")
        check(lib.lmx_decode(m._h, cache.seqs[0], 3 + i, 1, ptr(z), 1, stream_handle()), "lmx_decode")
        out.append(z)
    torch.cuda.synchronize()
    cache.close()
    return torch.cat(out)


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("dim", [40, 128, 200])
@pytest.mark.parametrize("ff", [33, 88, 8064, 8200])
def test_products_beside_each_other(cuda, dt, dim, ff):
    """Gate | up in less than one workgroup of 64 rows, in several, on the line between four rows a wave and two, and past it; experts of two layers, one behind latent attention."""
    cfg = config([delta(4, 2, dim, 40, 3, dense(ff)), delta(3, 3, 64, 48, 4, moe(72, 6, 2)), latent(3, 40, 20, 50, 36, 24, moe(40, 5, 3)), delta(4, 4, dim, dim, 4, dense(ff))], 136, 211)
    w = steady_routing(cfg, O.make_weights(cfg, 3, (18, 70)))
    m = build_config(cfg, w, DT[dt], 64)
    a = _steps(m, [5, 9, 2, 7, 1], 6)
    m.set_option("stack_fuse", 0)
    b = _steps(m, [5, 9, 2, 7, 1], 6)
    assert torch.isfinite(a.float()).all() and rel(a, b.double().cpu()) < TOL[dt] / 8


def test_a_shared_launch_is_a_group_of_its_own(cuda):
    """Launches by profile group, of 6 steps: what runs in a shared launch is under neither linear's own name."""
    cfg = config([delta(4, 2, 128, 40, 3, dense(88)), delta(3, 3, 64, 48, 4, moe(72, 6, 2)), latent(3, 40, 20, 50, 36, 24, moe(40, 5, 3)), delta(4, 4, 128, 128, 4, dense(88))], 136, 211)
    m = build_config(cfg, steady_routing(cfg, O.make_weights(cfg, 3, (18, 70))), torch.bfloat16, 64)
    names = ("decode.delta", "decode.delta_gate_up", "decode.gemv.gate_up", "decode.moe.gate_up", "decode.moe.gate_up_o", "decode.gemv.o")

    def launches():
        m.profile(True)
        _steps(m, [5, 9, 2, 7, 1], 6)
        prof = m.profile_read()
        m.profile(False)
        return [prof[k][1] if k in prof else 0 for k in names]
    assert launches() == [6, 12, 0, 0, 12, 12]
    m.set_option("stack_fuse", 0)
    assert launches() == [18, 0, 12, 12, 0, 24]


def _joined(m, steps):
    m.profile(True)
    out = _steps(m, [5, 9, 2, 7, 1], steps)
    prof = m.profile_read()
    m.profile(False)
    return out, tuple(prof[k][1] if k in prof else 0 for k in ("decode.delta_gate_up", "decode.moe.gate_up_o"))


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("width,heads,ff", [(1088, 17, 200), (2048, 32, 200), (2112, 33, 1500), (2112, 33, 9000), (4160, 4, 3200)])
def test_rows_of_several_loads(cuda, dt, width, heads, ff):
    """Rows of the gate | up shorter than, as long as and longer than what a wave has on the way, the last load in part; output projections of 3, 4 and 5 loads of two beside experts."""
    layers = [delta(2, 2, 64, 64, 4, dense(ff))] + ([delta(heads, heads, 64, 64, 4, moe(72, 6, 2))] if width <= 3072 else [])
    cfg = config(layers, width, 211)
    m = build_config(cfg, steady_routing(cfg, O.make_weights(cfg, 3, (18, 70))), DT[dt], 64)
    a, n = _joined(m, 4)
    assert n == (4, 4 if width <= 3072 else 0)
    m.set_option("stack_fuse", 0)
    b, n = _joined(m, 4)
    assert n == (0, 0) and torch.isfinite(a.float()).all() and rel(a, b.double().cpu()) < TOL[dt] / 8


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("N,H,act", [(8, 2048, 0), (2552, 2048, 0), (2560, 2048, 0), (2560, 3072, 0), (2552, 3072, 0), (2568, 3136, 0), (4088, 4096, 0), (4096, 4096, 0), (6136, 3136, 0),
                                     (6144, 3136, 0), (6152, 4096, 0), (2496, 2048, 3), (2560, 2048, 3), (4096, 2048, 0), (4104, 1544, 0), (5632, 2048, 3), (6144, 2048, 0), (6152, 2048, 0), (2560, 3136, 3), (6144, 4096, 3), (2560, 4160, 0)])
def test_the_row_and_its_linear(cuda, dt, N, H, act):
    from llava_mi355x import ops
    g = torch.Generator(device="cuda").manual_seed(N + H)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y, inj, post, pre = r(1, H), r(1, H).to(DT[dt]), r(1, H).to(DT[dt]), r(H).to(DT[dt]), r(H).to(DT[dt])
    w, b = (r(N, H) / H ** 0.5).to(DT[dt]), r(N).to(DT[dt])
    x1, xn = ops.residual_norm(x, y, post, inj, pre, 0.37, 1e-5, dtype=DT[dt])
    x2, one = ops.gemv_residual(x, y, post, inj, pre, w, 0.37, 1e-5, bias=b, act=act)
    z = xn.double() @ w.double().t() + b.double()
    if act:
        z = z.view(1, -1, 2, 32)
        z = (z[:, :, 0] * torch.sigmoid(z[:, :, 0]) * z[:, :, 1]).reshape(1, -1)
    assert rel(x2, x1.double().cpu()) < 1e-6 and rel(one, z.cpu()) < 2 * 2.0 ** (-8 if dt == "bf16" else -11)      # (an element of xn may round the other way)
