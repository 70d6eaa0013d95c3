"""What a cache holds behind the last key (an earlier request's values, with Inf and NaN among them) never reaches a later request: every attention kernel that reads whole tiles of
V^T clears it, because probability 0 times NaN is NaN.  The same launches on clean caches give the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["tiny", "tiny_gqa"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("context,rows", [(0, 1), (0, 100), (0, 700), (511, 1), (640, 33), (1343, 129), (700, 700)])
def test_a_sequence_after_one_of_nan(cuda, name, dt, context, rows):
    """A truncated sequence whose rows were all NaN, then a prompt in one or two portions (the second with key slices where it is short) and a step; the other one is fresh."""
    from llava_mi355x import _C
    from llava_mi355x.model import LmxKVCache
    from synthetic import build as harness, recipes as synth
    model = harness.build_model(synth.CONFIGS[name], dtype=dt, seed=0, max_position=2048)
    V = synth.CONFIGS[name].vocab_size
    g = torch.Generator().manual_seed(context + rows)
    emb = model.get_model().embed_tokens(torch.randint(3, V, (1, context + rows), generator=g).to(cuda))[0].contiguous()
    nan = torch.full((2000, emb.shape[1]), float("nan"), dtype=dt, device=cuda)
    outs = []
    for stale in (False, True):
        cache = LmxKVCache(model, 1)
        s = cache.seqs[0]
        if stale:
            _C.check(_C.lib.lmx_prefill(model._h, s, _C.ptr(nan), 2000, 0, None, 0, 1, _C.stream_handle()))
            _C.check(_C.lib.lmx_seq_truncate(s, 0, _C.stream_handle()))
        if context:
            _C.check(_C.lib.lmx_prefill(model._h, s, _C.ptr(emb), context, 0, None, 0, 1, _C.stream_handle()))
        got = torch.empty((rows, V), dtype=dt, device=cuda)
        _C.check(_C.lib.lmx_prefill(model._h, s, _C.ptr(emb[context:]), rows, 0, _C.ptr(got), 1, 1, _C.stream_handle()))
        step = torch.empty((1, V), dtype=dt, device=cuda)
        _C.check(_C.lib.lmx_decode(model._h, s, 5, 1, _C.ptr(step), 0, _C.stream_handle()))
        outs += [got, step]
    assert bool(outs[0].isfinite().all()) and torch.equal(outs[0], outs[2]) and torch.equal(outs[1], outs[3])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("form", ["causal", "whole", "window"])
@pytest.mark.parametrize("kv_len", [1, 7, 8, 63, 64, 65, 120, 129, 577])
def test_prompt_attention(cuda, dt, D, form, kv_len):
    from llava_mi355x import ops
    H, G, s_max = 4, 2, 640
    g = torch.Generator().manual_seed(kv_len)
    q_len = min(kv_len, 33)
    q = torch.randn(q_len, (H + 2 * G) * D, generator=g).to(dt).to(cuda)
    k, v = torch.randn(G, s_max, D, generator=g).to(dt), torch.randn(G, D, s_max, generator=g).to(dt)
    outs = []
    for stale in (False, True):
        k[:, kv_len:], v[:, :, kv_len:] = (float("nan"), float("inf")) if stale else (0, 0)
        kc, vt = k.to(cuda), v.to(cuda)
        if form == "window":
            outs.append(ops.window_attn(q, kc, vt, kv_len - q_len, H, G, D ** -0.5, window=50))
        else:
            outs.append(ops.flash_attn(q, kc, vt, q_len, kv_len, kv_len - q_len, H, G, D, form == "causal"))
    assert bool(outs[0].isfinite().all()) and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dt,D", [(torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128)])
def test_batched_steps(cuda, dt, D):
    from llava_mi355x import ops
    H, G, s_max, positions = 4, 2, 512, [0, 1, 63, 64, 127, 128, 200, 511]
    g = torch.Generator().manual_seed(D)
    qkv = torch.randn(len(positions), (H + 2 * G) * D, generator=g).to(dt).to(cuda)
    cs = torch.cat([torch.cos(torch.arange(s_max)[:, None] * torch.ones(D // 2)), torch.sin(torch.arange(s_max)[:, None] * torch.ones(D // 2))], 1).contiguous().to(cuda)
    k, v = torch.randn(G, s_max, D, generator=g).to(dt), torch.randn(G, D, s_max, generator=g).to(dt)
    words = [torch.tensor([p], dtype=torch.int32, device=cuda) for p in positions]
    outs = []
    for stale in (False, True):
        ks, vs = [], []
        for p in positions:
            kk, vv = k.clone(), v.clone()
            kk[:, p:], vv[:, :, p:] = (float("nan"), float("inf")) if stale else (0, 0)
            ks.append(kk.to(cuda)); vs.append(vv.to(cuda))
        outs.append(ops.decode_attn_batch(qkv, ks, vs, words, cs, H, G, D))
    assert bool(outs[0].isfinite().all()) and torch.equal(outs[0], outs[1])
