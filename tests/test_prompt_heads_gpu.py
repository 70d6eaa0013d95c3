"""Prompts of a layer-stack model read together: the last rows of the sequences that end in one piece share a product with the head and a launch of picks, 32 at a time
(csrc/stack.cpp, Model::stack_prefill)."""
import ctypes

import pytest
import torch

from test_vizosun_gpu import DT, TOL, model, oracle
from vizosun_util import tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("n", [1, 2, 32, 33, 35])
def test_picks_of_prompts_read_together(cuda, dt, n):
    """One row, a few, a full launch, and one and three rows past it: every sequence logs one token, whose score the oracle puts within rounding of the best."""
    from llava_mi355x._C import check, lib, stream_handle
    from llava_mi355x.engine_lm import LmxKVCache
    m = model("mixed", dt)
    ts = [tokens("mixed", 3 + i % 5, 200 + i) for i in range(n)]
    caches = [LmxKVCache(m, 1) for _ in ts]
    embeds = m.get_model().embed_tokens(torch.tensor([x for t in ts for x in t], device=cuda)).split([len(t) for t in ts])
    check(lib.lmx_prefill_batch(m._h, (ctypes.c_void_p * n)(*[c.seqs[0].value for c in caches]), n, (ctypes.c_void_p * n)(*[e.data_ptr() for e in embeds]),
                                (ctypes.c_int32 * n)(*[len(t) for t in ts]), 0, 1, stream_handle()), "lmx_prefill_batch")
    for t, c in zip(ts, caches):
        host, got = (ctypes.c_int64 * 4)(), ctypes.c_int32(0)
        check(lib.lmx_seq_read_tokens(c.seqs[0], host, 4, ctypes.byref(got), stream_handle()), "lmx_seq_read_tokens")
        z = oracle("mixed", t, dt)[-1].double()
        assert got.value == 1 and z[host[0]] >= z.max() - 2 * TOL[dt] * z.norm(), (t, host[0])
        c.close()


@pytest.mark.parametrize("variant", [30, 881])
def test_picks_whatever_tile_the_linears_are_told(cuda, variant):
    """gemm_variant names a tile of 16-bit output for the prompt's linears; the head's product, with fp32 output, is not one of them."""
    from llava_mi355x._C import check, lib, stream_handle
    from llava_mi355x.engine_lm import LmxKVCache
    from llava_mi355x.vizosun import VizosunConfig, VizosunForCausalLM
    from vizosun_util import CONFIGS, weights
    name, dt, n = "odd", "bf16", 3
    w = weights(name, steady=True)
    m = VizosunForCausalLM(VizosunConfig.from_dict(CONFIGS[name], {k: tuple(v.shape) for k, v in w.items()}), dtype=DT[dt], max_position=128, gemm_variant=variant).load_state_dict(w)
    ts = [tokens(name, 9 + i, 300 + i) for i in range(n)]
    caches = [LmxKVCache(m, 1) for _ in ts]
    embeds = m.get_model().embed_tokens(torch.tensor([x for t in ts for x in t], device=cuda)).split([len(t) for t in ts])
    check(lib.lmx_prefill_batch(m._h, (ctypes.c_void_p * n)(*[c.seqs[0].value for c in caches]), n, (ctypes.c_void_p * n)(*[e.data_ptr() for e in embeds]),
                                (ctypes.c_int32 * n)(*[len(t) for t in ts]), 0, 1, stream_handle()), "lmx_prefill_batch")
    for t, c in zip(ts, caches):
        host, got = (ctypes.c_int64 * 4)(), ctypes.c_int32(0)
        check(lib.lmx_seq_read_tokens(c.seqs[0], host, 4, ctypes.byref(got), stream_handle()), "lmx_seq_read_tokens")
        z = oracle(name, t, dt)[-1].double()
        assert got.value == 1 and z[host[0]] >= z.max() - 2 * TOL[dt] * z.norm(), (t, host[0])
        c.close()
