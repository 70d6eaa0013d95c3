"""What a cache holds behind the last key (an earlier request's values, with Inf and NaN among them) never reaches a later request, although probability 0 times NaN is NaN: the launches
that append a portion's rows clear V^T to the end of the last row's 64 keys, and the kernels of a step clear what they loaded.  The same launches on clean caches give the same
bits."""
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


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_a_layer_stack_sequence_after_one_of_nan(cuda, dt):
    """The same for windowed layers: widths with and without whole rotation groups, windows that end inside a tile."""
    from llava_mi355x import _C
    from llava_mi355x.engine_lm import LmxKVCache
    from siterax_util import build, tokens
    for name in ("mixed", "odd"):
        m = build(name, dt)
        for n, more in ((2, 0), (70, 9), (129, 60)):
            ids = torch.tensor([tokens(name, n + more + 1, n)], device=cuda)
            outs = []
            for stale in (False, True):
                first = LmxKVCache(m, 1)
                if stale:
                    nan = torch.full((400, m.row_pitch), float("nan"), dtype=dt, device=cuda)
                    _C.check(_C.lib.lmx_prefill(m._h, first.seqs[0], _C.ptr(nan), 400, 0, None, 0, 1, _C.stream_handle()))
                _C.check(_C.lib.lmx_seq_truncate(first.seqs[0], 0, _C.stream_handle()))
                o = m.forward(ids[:, :n], past_key_values=first)
                got = [o.logits]
                if more:
                    got.append(m.forward(ids[:, n:n + more], past_key_values=first).logits)
                got.append(m.forward(ids[:, n + more:], past_key_values=first).logits)
                outs.append(got)
            for a, b in zip(*outs):
                assert bool(a.isfinite().all()) and torch.equal(a, b), (name, n, more)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,pos0", [(1, 0), (63, 0), (64, 0), (65, 8), (70, 56), (130, 120), (1, 255), (100, 156)])
def test_appended_rows_clear_the_rest_of_their_tile(cuda, dt, D, T, pos0):
    """rope_kv: V^T from the last row to the end of its 64 keys is 0, what lies before the portion and behind that tile stays."""
    from llava_mi355x import ops
    H, G, s_max = 2, 2, 256
    g = torch.Generator().manual_seed(T + pos0)
    qkv = torch.randn(T, (H + 2 * G) * D, generator=g).to(dt).to(cuda)
    v = qkv[:, (H + G) * D:].reshape(T, G, D).permute(1, 2, 0).clone()
    kc, vt = torch.zeros(G, s_max, D, dtype=dt, device=cuda), torch.full((G, D, s_max), float("nan"), dtype=dt, device=cuda)
    ops.rope_kv(qkv, kc, vt, torch.ones(s_max, D, device=cuda), pos0, H, G, D)
    end = pos0 + T
    whole = -(-end // 64) * 64
    assert torch.equal(vt[:, :, pos0:end], v) and not bool(vt[:, :, end:whole].any())
    assert bool(vt[:, :, :pos0].isnan().all()) and bool(vt[:, :, whole:].isnan().all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,H,G,T,pos0", [(128, 32, 32, 1087, 0), (128, 16, 16, 2000, 40), (64, 64, 16, 2001, 8), (128, 32, 32, 1088, 64)])
def test_the_fused_projection_clears_it_too(cuda, dt, D, H, G, T, pos0):
    from llava_mi355x import ops
    s_max, K = 2176, 128
    x, w = torch.randn(T, K, device=cuda).to(dt), torch.randn((H + 2 * G) * D, K, device=cuda).to(dt)
    out = torch.empty(T, (H + 2 * G) * D, dtype=dt, device=cuda)
    kc, vt = torch.zeros(G, s_max, D, dtype=dt, device=cuda), torch.full((G, D, s_max), float("nan"), dtype=dt, device=cuda)
    ops.gemm_qkv_rope(x, w, out, kc, vt, torch.ones(s_max, D, device=cuda), pos0, H, G, D)
    end = pos0 + T
    whole = -(-end // 64) * 64
    assert bool(vt[:, :, pos0:end].isfinite().all()) and not bool(vt[:, :, end:whole].any())
    assert bool(vt[:, :, :pos0].isnan().all()) and bool(vt[:, :, whole:].isnan().all())


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
