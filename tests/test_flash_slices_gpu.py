"""A short prompt portion on a long context: its attention's keys are cut into slices over the workgroups and merged by a second launch (csrc/attention.hip: flash_slices,
flash_merge_kernel).  Every row against the one-token step of the same position (another kernel, its own merge), for contexts at the borders of the slices' tiles, one row
and more than one query block, heads of 128 and, two to a kv head, of 64; the tolerance is that of the other comparisons of two 16-bit forms of one step."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("context,rows", [(511, 1), (448, 64), (640, 33), (1343, 129), (1919, 5)])
@pytest.mark.parametrize("name", ["tiny", "tiny_gqa"])
def test_rows_of_a_portion_as_single_steps(cuda, name, dt, context, rows):
    from llava_mi355x import _C
    from llava_mi355x.model import LmxKVCache
    from synthetic import build as harness, recipes as synth
    cfg = synth.CONFIGS[name]
    model = harness.build_model(cfg, dtype=dt, seed=0, max_position=2048)
    torch.manual_seed(context)
    V = cfg.vocab_size
    ids = torch.randint(3, V, (1, context + rows), device=cuda)
    emb = model.get_model().embed_tokens(ids)[0].contiguous()
    caches = [LmxKVCache(model, 1), LmxKVCache(model, 1)]
    for c in caches:
        _C.check(_C.lib.lmx_prefill(model._h, c.seqs[0], _C.ptr(emb), context, 0, None, 0, 1, _C.stream_handle()))
    got = torch.empty((rows, V), dtype=dt, device=cuda)
    _C.check(_C.lib.lmx_prefill(model._h, caches[0].seqs[0], _C.ptr(emb[context:]), rows, 0, _C.ptr(got), 1, 1, _C.stream_handle()))
    want = torch.empty((rows, V), dtype=dt, device=cuda)
    for i in range(rows):
        _C.check(_C.lib.lmx_decode(model._h, caches[1].seqs[0], int(ids[0, context + i]), 1, _C.ptr(want[i:]), 0, _C.stream_handle()))
    assert (got.float() - want.float()).abs().max().item() <= 2e-2 * max(1.0, want.float().abs().max().item())
