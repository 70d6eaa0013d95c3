"""The K slices of a prompt's q|k|v, o and down linears added by the launch that reads their rows (csrc/elementwise.hip: rope_kv_kernel over slices; csrc/gemm_rows.hip:
rows_reduce_norm_kernel) against a reduction launch and then rope_kv / rmsnorm: the same additions in the same order, rounded where the stored row would be, the norm's sum in
rmsnorm_reg_kernel's order, so logits, hidden states and generated ids (which read the caches) are BIT-IDENTICAL.  7B and 13B widths (two and three chunks a thread), both
16-bit types, row counts at the edges of a 64-row cache block and of the row tiles, and a chunked prompt; 700 rows bring no slices and run as before."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,dtype,rows,kw", [
    ("llava15_7b", torch.bfloat16, 33, {}), ("llava15_7b", torch.bfloat16, 64, {}), ("llava15_7b", torch.float16, 65, {}), ("llava15_7b", torch.bfloat16, 139, {}), ("llava15_7b", torch.float16, 256, {}),
    ("llava15_13b", torch.bfloat16, 97, {}), ("llava15_13b", torch.float16, 139, {}), ("llava15_7b", torch.bfloat16, 257, {"prefill_chunk": 128}), ("llava15_7b", torch.bfloat16, 700, {})])
def test_slices_added_by_their_reader(cuda, name, dtype, rows, kw):
    from synthetic import build as harness, recipes as synth
    cfg = synth.with_layers(synth.CONFIGS[name], 3, 1)
    model = harness.build_model(cfg, dtype=dtype, seed=0, device_rng=True, max_position=2048)
    ids = torch.from_numpy(synth.make_prompt(cfg, rows, image_positions=(), seed=rows))[None].to(cuda)

    def run(on):
        model.set_option("fuse_slices", on)
        try:
            out = model.forward(input_ids=ids, use_cache=True, output_hidden_states=True)
            logits, hidden = out.logits.clone(), [t.clone() for t in out.hidden_states]
            out.past_key_values.close()
            return logits, hidden, model.generate(inputs=ids, do_sample=False, max_new_tokens=4, eos_token_id=-1, **kw)
        finally:
            model.set_option("fuse_slices", 1)

    la, ha, ga = run(1)
    lb, hb, gb = run(0)
    assert torch.isfinite(la).all() and torch.equal(la, lb) and torch.equal(ga, gb)
    assert all(torch.equal(a, b) for a, b in zip(ha, hb))
