"""One sequence's decode step whose attention runs in splits: the output projection adds them (csrc/gemv2.h: SPLITS) against the attention's own merge and the oracle.  Two to sixteen splits
and more, windows on a few of them, gates and sinks, rows of up to the 4096 a workgroup holds and past it, outputs below and above a row a wave; the projection
itself on given splits against float64."""
import pytest
import torch

from oracle import siterax_oracle as O
from siterax_util import CONFIGS, config, layer, rel, tokens

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16}
TOL = {"bf16": 4e-2, "f16": 6e-3}
AT = (127, 128, 300, 511, 700, 897, 1024, 2046, 2100)
FORMS = {
    "mixed": CONFIGS["mixed"], "wide": CONFIGS["wide"],
    "full": config([layer(32, 4, 128, 128, 0, 64, 64)], 2056, 64, None),       # 4096 inputs, two rows a wave
    "ten": config([layer(24, 3, 128, 128, 0, 64, 64)], 2056, 64, None),        # 3072 inputs, two rows a wave: ten splits at most
    "past": config([layer(33, 3, 128, 128, 0, 64, 64)], 96, 64, None),         # 4224 inputs: the attention merges
}


def steps(m, toks):
    """logits of two steps behind every length of AT"""
    from llava_mi355x.engine_lm import LmxKVCache
    out = []
    for n in AT:
        r = m.forward(torch.tensor([toks[:n]], device=m.device))
        for i in range(2):
            r = m.forward(torch.tensor([toks[n + i:n + i + 1]], device=m.device), past_key_values=r.past_key_values)
            out.append(r.logits[0, -1])
        torch.cuda.synchronize()
        r.past_key_values.close()
    return torch.stack(out)


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("name", list(FORMS))
def test_splits_added_by_the_projection(cuda, name, dt):
    from llava_mi355x.siterax import SiteraxConfig, SiteraxForCausalLM
    cfg = FORMS[name]
    w = O.make_weights(cfg, 1)
    m = SiteraxForCausalLM(SiteraxConfig.from_dict(cfg), dtype=DT[dt], max_position=2176).load_state_dict(w)
    g = torch.Generator().manual_seed(9)
    toks = torch.randint(0, cfg["vocab"], (AT[-1] + 2,), generator=g).tolist()
    want = O.logits(cfg, w, toks)[[n + i for n in AT for i in range(2)]]
    a = steps(m, toks)
    m.set_option("stack_fuse", 0)
    b = steps(m, toks)
    assert rel(a, want) < TOL[dt] and rel(a, b.double().cpu()) < TOL[dt] / 2


def merged(p, gate, sink):
    """the row that partials stand for, in float64"""
    p = p.double()
    D = p.shape[2] - 4
    m = p[:, :, D]
    M = m.max(1, keepdim=True).values.clamp_min(0.0 if sink else -float("inf"))
    w = torch.exp2(m - M)
    x = (w[:, :, None] * p[:, :, :D]).sum(1) / ((w * p[:, :, D + 1]).sum(1, keepdim=True) + (torch.exp2(-M) if sink else 0.0))
    return (x if gate is None else x * torch.sigmoid(gate.double())[:, None]).reshape(-1)


def partials(heads, n_split, D, g):
    """maxima some powers of two apart, sums as of a few dozen keys; what follows a row's sum is nobody's"""
    p = torch.randn(heads, n_split, D + 4, generator=g)
    l = 1 + 40 * torch.rand(heads, n_split, generator=g)
    p[:, :, :D] *= l[:, :, None]
    p[:, :, D], p[:, :, D + 1], p[:, :, D + 2:] = 6 * torch.randn(heads, n_split, generator=g), l, float("nan")
    return p


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("heads,D,N,splits", [(8, 128, 200, range(2, 17)), (1, 64, 9, (2, 16)), (3, 256, 2050, (5, 11, 16)), (16, 256, 2056, (2, 7, 8)), (24, 128, 2049, (3, 9, 10)), (32, 128, 97, (4, 8)), (5, 64, 4100, (6, 13))])
def test_given_splits_against_float64(cuda, dt, heads, D, N, splits):
    from llava_mi355x import ops
    g = torch.Generator().manual_seed(heads * D + N)
    w = (torch.randn(N, heads * D, generator=g) / (heads * D) ** 0.5).to(DT[dt])
    for n in splits:
        p, gate, sink = partials(heads, n, D, g), (torch.randn(heads, generator=g) if n % 2 else None), n % 3 == 0
        if n > 2:                                            # a split whose keys the window has left
            p[::2, 1, :D], p[::2, 1, D], p[::2, 1, D + 1] = 0, -float("inf"), 0
        gate = None if gate is None else gate.to(DT[dt])
        got = ops.gemv_heads(p.to(cuda), w.to(cuda), None if gate is None else gate.to(cuda), sink)[0].double().cpu()
        x = merged(p, gate, sink)
        want, absolute = w.double() @ x, w.double().abs() @ x.abs()
        # the row and the output are rounded once each: at most 2^-9 (bf16) or 2^-12 (f16) off, relative; 1e-5 for the fp32 weights, sums of 17 terms and products
        half = 2.0 ** -9 if dt == "bf16" else 2.0 ** -12
        assert bool(((got - want).abs() <= 1.01 * (absolute * (half + 1e-5) + want.abs() * half) + 1e-6).all()), (n, ((got - want).abs() / absolute).max().item())


@pytest.mark.parametrize("n", [3, 5, 7, 9])
def test_an_infinite_value_stays_one(cuda, n):
    """Forms for more splits than there are read the last one more than once: it weighs nothing the second time, whatever it holds."""
    from llava_mi355x import ops
    g = torch.Generator().manual_seed(n)
    p, w = partials(4, n, 64, g), torch.randn(40, 256, generator=g).bfloat16()
    p[2, n - 1, 5] = float("inf")
    w[w == 0] = 1
    got = ops.gemv_heads(p.to(cuda), w.to(cuda))[0].cpu()
    assert torch.equal(got.float(), torch.where(w[:, 2 * 64 + 5] > 0, float("inf"), -float("inf")))
