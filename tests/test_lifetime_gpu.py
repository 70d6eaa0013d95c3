"""Sequences and their model go in any order: a garbage collector that takes both (a traceback that held them) runs their finalizers in an order of its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("used", [False, True])
def test_sequences_outlive_their_model(cuda, used):
    from llava_mi355x import _C
    from llava_mi355x.model import LmxKVCache
    from synthetic import build as harness, recipes as synth
    cfg = synth.CONFIGS["tiny"]
    model = harness.build_model(cfg, dtype=torch.bfloat16, seed=0)
    caches = [LmxKVCache(model, 2), LmxKVCache(model, 1)]
    emb = model.get_model().embed_tokens(torch.arange(3, 12, device=cuda)[None])[0].contiguous()
    if used:
        for s in caches[0].seqs:
            _C.check(_C.lib.lmx_prefill(model._h, s, _C.ptr(emb), 9, 0, None, 0, 1, _C.stream_handle()))
    caches[1].close()                                     # into the model's pool
    h, model._h = model._h, None
    _C.check(_C.lib.lmx_destroy(h))
    left, caches[0].seqs = caches[0].seqs, []
    assert _C.lib.lmx_seq_truncate(left[0], 0, _C.stream_handle()) != 0      # refused, the model is gone
    assert _C.lib.lmx_seq_copy(left[0], left[1], _C.stream_handle()) != 0
    for s in left:
        _C.check(_C.lib.lmx_seq_destroy(s))
    model = harness.build_model(cfg, dtype=torch.bfloat16, seed=0)           # and the next model's sequences are its own
    c = LmxKVCache(model, 1)
    _C.check(_C.lib.lmx_prefill(model._h, c.seqs[0], _C.ptr(emb), 9, 0, None, 0, 1, _C.stream_handle()))
    assert _C.lib.lmx_seq_length(c.seqs[0]) == 9
