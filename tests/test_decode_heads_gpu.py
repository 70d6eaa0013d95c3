"""One sequence's decode step whose attention runs in splits: the output projection adds them (csrc/gemv2.h: SPLITS) against the attention's own merge and the oracle.  Two to sixteen splits
and more, windows on a few of them, gates and sinks, rows of up to the 4096 a workgroup holds and past it, outputs below and above a row a wave."""
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
