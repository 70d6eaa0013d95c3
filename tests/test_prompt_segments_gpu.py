"""Prompts of a layer-stack model read together: norms, rotations, caches and attention of the rows of up to 32 sequences in one launch (csrc/stack.cpp Model::stack_prefill, csrc/stack_mixers.cpp
Model::stack_mix_prefill).  Lengths around the 64-row blocks and 32-key tiles, more sequences than one launch takes, sequences that go on beside new ones."""
import pytest
import torch

import test_siterax_gpu as siterax
import test_vizosun_gpu as vizosun

pytestmark = pytest.mark.gpu


def read(m, caches, portions):
    emb = [m.get_model().embed_tokens(torch.tensor(p)) for p in portions]
    got = m.prefill_logits(caches, emb, [list(range(len(p))) for p in portions])
    torch.cuda.synchronize()
    return [g[:, : m.config.vocab_size] for g in got.split([len(p) for p in portions])]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("family,name", [(siterax, "mixed"), (siterax, "odd"), (siterax, "single"), (vizosun, "mixed"), (vizosun, "plain"), (vizosun, "single"), (vizosun, "many")])
def test_rows_of_several_sequences(cuda, family, name, dt):
    from llava_mi355x.engine_lm import LmxKVCache
    m = family.model(name, dt)
    oracle = (lambda t: vizosun.oracle(name, t, dt)) if family is vizosun else (lambda t: siterax.oracle(name, t))
    first, then = [1, 31, 32, 33, 63, 64, 65, 97, 128, 129, 200], [3, 64, 1, 40]
    ts = [family.tokens(name, n + (then[i] if i < len(then) else 0), 400 + i) for i, n in enumerate(first)]
    caches = [LmxKVCache(m, 1) for _ in ts]
    rows = read(m, caches, [t[:n] for t, n in zip(ts, first)])
    new = family.tokens(name, 66, 430)                      # four sequences go on in one call with a new one
    caches.append(LmxKVCache(m, 1))
    more = read(m, caches[:len(then)] + caches[-1:], [t[n:] for t, n in zip(ts, first[:len(then)])] + [new])
    for i, g in enumerate(more[:-1]):
        rows[i] = torch.cat([rows[i], g])
    assert max(family.rel(g, oracle(t)) for t, g in zip(ts + [new], rows + more[-1:])) < family.TOL[dt]
    for c in caches:
        c.close()


@pytest.mark.parametrize("family", [siterax, vizosun])
def test_more_sequences_than_one_launch_takes(cuda, family):
    from llava_mi355x.engine_lm import LmxKVCache
    m = family.model("mixed", "bf16")
    ts = [family.tokens("mixed", 2 + (7 * i) % 70, 500 + i) for i in range(35)]
    caches = [LmxKVCache(m, 1) for _ in ts]
    rows = read(m, caches, ts)
    oracle = (lambda t: vizosun.oracle("mixed", t, "bf16")) if family is vizosun else (lambda t: siterax.oracle("mixed", t))
    assert max(family.rel(g, oracle(t)) for t, g in zip(ts, rows)) < family.TOL["bf16"]
    for c in caches:
        c.close()


@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_chosen_rows_of_several_sequences(cuda, dt):
    """Single rows (more than a gather takes), pairs, whole stretches and a sequence without any, in one call: the rows of the call that asks for all of them."""
    from llava_mi355x.engine_lm import LmxKVCache
    m = siterax.model("mixed", dt)
    n = [129, 70, 1, 200, 33]
    ts = [siterax.tokens("mixed", k, 600 + i) for i, k in enumerate(n)]
    chosen = [list(range(0, 129, 2)), [0, 1, 7, 8, 69], [0], list(range(10, 75)) + [199], [31, 32]]
    oracle = [siterax.oracle("mixed", t) for t in ts]
    caches = [LmxKVCache(m, 1) for _ in ts]
    got = m.prefill_logits(caches, [m.get_model().embed_tokens(torch.tensor(t)) for t in ts], chosen)
    torch.cuda.synchronize()
    got = got[:, : m.config.vocab_size].split([len(c) for c in chosen])
    assert max(siterax.rel(g, o[c]) for g, o, c in zip(got, oracle, chosen)) < siterax.TOL[dt]
    for c in caches:
        c.close()


@pytest.mark.parametrize("name", ["plain", "mixed"])
def test_more_rows_than_the_latents_expand_at_once(cuda, name):
    """9000 rows of new prompts: the first 20 of them together, the 21st would pass 8192 rows."""
    from llava_mi355x.engine_lm import LmxKVCache
    m = vizosun.model(name, "bf16")
    n = [400] * 20 + [300, 390, 310]
    ts = [vizosun.tokens(name, k, 700 + i) for i, k in enumerate(n)]
    caches = [LmxKVCache(m, 1) for _ in ts]
    rows = read(m, caches, ts)
    for c in caches:
        c.close()
    assert max(vizosun.rel(rows[i], vizosun.oracle(name, ts[i], "bf16")) for i in (0, 19, 20, 21, 22)) < vizosun.TOL["bf16"]
