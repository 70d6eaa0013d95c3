"""The K slices of a prompt's linears added by the launch that reads their rows, at the shapes test_fuse_slices_gpu.py does not reach: later portions behind cached rows, prompts of up to
32 rows, grouped-query and 64-wide heads (csrc/elementwise.hip: rope_kv_kernel over slices), and a tensor-parallel rank, whose q|k|v alone stays in slices.  Every case says which linears
come in slices there, asked of the library, so that a change of its forms shows.  Bits: logits of every row, of three decode steps behind them, and the caches by what those steps read."""
import ctypes
from dataclasses import replace

import pytest
import torch

pytestmark = pytest.mark.gpu
HOOK_T = ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_uint64, ctypes.c_int32, ctypes.c_void_p, ctypes.c_void_p)

# widths, heads of q and of k / v; portions of the prompt; per portion which of q|k|v, o, down come in slices
CASES = [("7b", 4096, 11008, 32, 32, (139, 139), ("qd", "qd")), ("7b", 4096, 11008, 32, 32, (256, 131), ("qd", "qd")), ("13b", 5120, 13824, 40, 40, (139, 200), ("qd", "qd")),
         ("7b", 4096, 11008, 32, 32, (2, 20, 7), ("od", "od", "od")), ("gqa", 4096, 4096, 32, 8, (64, 17, 300), ("qod", "qod", "qod")), ("gqa", 4096, 4096, 32, 8, (139, 3), ("", "qod")),
         ("d64", 2560, 2560, 40, 40, (64, 33), ("qod", "qod")), ("d64", 2560, 2560, 40, 40, (300, 64), ("q", "qod")), ("gqa64", 2560, 2560, 40, 10, (100, 28, 65), ("qod", "qod", "qod"))]


def _bits(model, portions, on):
    from llava_mi355x._C import check, lib, ptr, stream_handle
    from llava_mi355x.engine_lm import LmxKVCache
    model.set_option("fuse_slices", on)
    cache, out, V = LmxKVCache(model, 1), [], model._vocab_cap
    e = model.get_model().embed_tokens(torch.arange(5, 5 + sum(portions), device="cuda"))
    at = 0
    for n in portions:
        z = torch.empty((n, V), dtype=model.dtype, device="cuda")
        check(lib.lmx_prefill(model._h, cache.seqs[0], ptr(e[at:at + n].contiguous()), n, 0, ptr(z), 1, 1, stream_handle()), "lmx_prefill")
        out.append(z); at += n
    for t in (3, 11, 17):
        z = torch.empty((1, V), dtype=model.dtype, device="cuda")
        check(lib.lmx_decode(model._h, cache.seqs[0], t, 1, ptr(z), 1, stream_handle()), "lmx_decode")
        out.append(z)
    torch.cuda.synchronize()
    cache.close()
    model.set_option("fuse_slices", 1)
    return torch.cat(out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name,H,I,nh,nkv,portions,sliced", CASES)
def test_portions(cuda, dtype, name, H, I, nh, nkv, portions, sliced):
    from llava_mi355x import ops
    from synthetic import build as harness, recipes as synth
    cfg = replace(synth.with_layers(synth.CONFIGS["llava15_7b"], 3, 1), hidden_size=H, intermediate_size=I, num_attention_heads=nh, num_key_value_heads=nkv, vocab_size=1024)
    D = H // nh
    for n, want in zip(portions, sliced):
        got = "".join(c for c, N, K in (("q", (nh + 2 * nkv) * D, H), ("o", H, H), ("d", H, I)) if ops.gemm_form(dtype, n, N, K)[0] == 1 and ops.gemm_form(dtype, n, N, K)[3] > 1)
        assert got == want, (n, got)
    model = harness.build_model(cfg, dtype=dtype, seed=0, device_rng=True, max_position=1024)
    a, b = _bits(model, portions, 1), _bits(model, portions, 0)
    assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("world,rows", [(2, 64), (4, 100)])
def test_a_rank(cuda, world, rows):
    """One rank's partial sums: o and down end in the sum over ranks, q|k|v does not."""
    from llava_mi355x import _C, ops
    from synthetic import build as harness, recipes as synth
    cfg = replace(synth.with_layers(synth.CONFIGS["llava15_7b"], 2, 1), vocab_size=1024)
    assert ops.gemm_form(torch.bfloat16, rows, 3 * cfg.hidden_size // world, cfg.hidden_size)[3] > 1
    noop = HOOK_T(lambda buf, count, dt, stream, ctx: None)
    model = harness.build_model(cfg, dtype=torch.bfloat16, seed=0, device_rng=True, max_position=512, tp_rank=0, tp_world=world)
    _C.check(_C.lib.lmx_tp_set_allreduce_hook(model._h, ctypes.cast(noop, ctypes.c_void_p), None))
    a, b = _bits(model, (rows, rows), 1), _bits(model, (rows, rows), 0)
    assert torch.isfinite(a).all() and torch.equal(a, b)
