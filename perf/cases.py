"""What a program built on this package has it do, as timed cases: image encoding, prompts, conversation turns, single-request and batched decoding and the training step
of LLaVA-1.5, and prompts and decoding of the two layer-stack families, each through the public entry points, with a plain float64 computation of the same results.

Sizes are those of LLaVA-1.5-7B / 13B and of the layer-stack sizes of bench.py; the depth of a drawn model is smaller.  Weights are random and laid out like a trained model's
in the two ways that matter here: a sublayer adds little to the stream, and the next token is clear (the head answers every token with one other, see `successor`), so greedy
ids are the same in 16 and in 64 bits."""
from __future__ import annotations

import ctypes
import gc
import math
import os
import sys
import zlib

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llava-plus-codebase_amd"))

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
VOCAB = 32000
LLAVA = {4096: (32, 11008), 5120: (40, 13824)}                                       # width: heads (of 128), feed-forward width
VIS = {"width": 1024, "ff": 4096, "heads": 16, "layers": 24, "run": 23, "size": 336, "patch": 14, "tokens": 576}     # CLIP ViT-L/14-336, features of layer -2
SITERAX = {2048: (16, 4, 128, 5632), 3072: (32, 8, 96, 8192), 4096: (32, 8, 128, 11008)}          # width: heads, kv heads, head width, feed-forward width
VIZOSUN = {2048: (16, 128, 768, 512, 5632, 1408), 4096: (32, 128, 1536, 512, 11008, 2752)}       # width: heads, head width, query latent, kv latent, ff, expert ff
EXPERTS, TOP, RANK, BUCKETS, MUL = 16, 4, 128, 8191, (137, 3)
EPS = 1e-5
IMAGE = -200                                                                         # marker of an image in a prompt


def listed():
    return [
        # the first answer of a conversation up to its first token: one photo and a 511-token prompt (1087 positions), the whole of LLaVA-1.5-7B
        {"name": "chat_prompt", "op": "llava_prompt", "dtype": "bf16", "width": 4096, "layers": 32, "images": 1, "rows": 511},
        # a later turn of the tool loop: the earlier turns are cached, the tool's answer follows
        {"name": "chat_turn", "op": "llava_turn", "dtype": "f16", "width": 4096, "layers": 32, "context": 1208, "rows": 139},
        # the crops of one high-resolution picture, or the pictures of requests that arrived together
        {"name": "images", "op": "llava_images", "dtype": "f16", "width": 4096, "images": 4},
        # one user reading along: greedy tokens behind the prompt of the first case
        {"name": "chat_decode", "op": "llava_decode", "dtype": "bf16", "width": 4096, "layers": 32, "requests": 1, "context": 1087, "tokens": 16},
        # a served model with sixteen conversations of different lengths in flight
        {"name": "chat_batch", "op": "llava_decode", "dtype": "bf16", "width": 4096, "layers": 32, "requests": 16, "context": 1087, "tokens": 8},
        # one visual-instruction-tuning step over samples of unequal length (two layers of the model's width: the step's cost is the layers' sum)
        {"name": "train_step", "op": "llava_train", "dtype": "bf16", "width": 4096, "layers": 2, "samples": 4, "rows": 2048},
        # a long document read by the smaller layer-stack model
        {"name": "siterax_prompt", "op": "siterax_prompt", "dtype": "bf16", "width": 2048, "layers": 12, "window": 0, "requests": 1, "rows": 2048},
        # its answer, token by token: the smallest calls
        {"name": "siterax_decode", "op": "siterax_decode", "dtype": "bf16", "width": 2048, "layers": 12, "window": 0, "requests": 1, "context": 601, "tokens": 32},
        # offline generation over 32 documents with a windowed model
        {"name": "siterax_batch", "op": "siterax_decode", "dtype": "bf16", "width": 4096, "layers": 12, "window": 1024, "requests": 32, "context": 1300, "tokens": 8},
        # three prompts of unequal length read together
        {"name": "vizosun_prompt", "op": "vizosun_prompt", "dtype": "bf16", "width": 2048, "layers": 12, "window": 1024, "requests": 3, "rows": 1100},
        # a short question and its answer
        {"name": "vizosun_request", "op": "vizosun_request", "dtype": "bf16", "width": 2048, "layers": 12, "window": 1024, "requests": 1, "rows": 45, "tokens": 32},
        # 32 short questions answered together
        {"name": "vizosun_batch", "op": "vizosun_request", "dtype": "bf16", "width": 4096, "layers": 12, "window": 1024, "requests": 32, "rows": 64, "tokens": 8},
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    op = rng.choice(["llava_prompt", "llava_turn", "llava_images", "llava_decode", "llava_train", "siterax_prompt", "siterax_decode", "vizosun_prompt", "vizosun_request"])
    c = {"op": op, "dtype": rng.choice(["bf16", "f16"])}
    if op.startswith("llava"):
        c["width"] = rng.choice([4096, 4096, 5120])
        c["layers"] = rng.randint(2, 6)
        if op == "llava_prompt":
            c.update(images=rng.randint(0, 2), rows=log(24, 1100))
        elif op == "llava_turn":
            c.update(context=log(64, 1400), rows=log(2, 600))
        elif op == "llava_images":
            del c["layers"]
            c.update(images=log(1, 8))
        elif op == "llava_decode":
            c.update(requests=log(1, 32), context=log(16, 1500), tokens=rng.randint(4, 12))
        else:
            c.update(dtype="bf16", width=4096, layers=1, samples=rng.randint(1, 4), rows=log(700, 2000))
        return c
    c.update(dtype="bf16", width=rng.choice([2048, 3072, 4096] if op.startswith("siterax") else [2048, 4096]), layers=rng.choice([4, 8]), window=rng.choice([0, 1024]),
             requests=log(1, 4) if op.endswith("prompt") else log(1, 32))
    if op.endswith("prompt"):
        c["rows"] = log(60, 2048 if c["requests"] == 1 else 900)
    elif op == "siterax_decode":
        c.update(context=log(16, 1900), tokens=rng.randint(4, 24))
    else:
        c.update(rows=log(5, 70), tokens=rng.randint(4, 24))
    return c


def lengths(case, longest):
    """Rows of each request: unequal, the first the longest."""
    n = case.get("requests", case.get("samples", 1))
    return [max(2, longest - longest * 9 * i // (16 * n) - i % 3) for i in range(n)]


# ---- inputs -------------------------------------------------------------------------------------------------------------------------------------

def seeded(seed, name):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFF)


def normal(seed, name, shape, std, dtype, mean=0.0):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=seeded(seed, name))


def successor(seed):
    """successor[t]: the token that follows t."""
    return torch.randperm(VOCAB, generator=seeded(seed, "successor"), device="cuda")


def prompt(seed, n, name):
    return torch.randint(3, VOCAB, (n,), generator=seeded(seed, "prompt " + name), device="cuda")


def chain(seed, first, n):
    """The n tokens that follow each of `first`."""
    nxt, out = successor(seed), []
    for _ in range(n):
        first = nxt[first]
        out.append(first)
    return torch.stack(out)


def head_like(seed, embed):
    """Head rows that answer every token's embedding with its successor."""
    head = torch.empty_like(embed)
    head[successor(seed)] = embed
    return head * embed.shape[1] ** -0.5


def llava_shapes(case):
    W, (_, F) = case["width"], LLAVA[case["width"]]
    s = {"model.embed_tokens.weight": (VOCAB, W), "lm_head.weight": (VOCAB, W), "model.norm.weight": (W,)}
    for i in range(case.get("layers", 1)):
        p = f"model.layers.{i}."
        s.update({p + f"self_attn.{n}_proj.weight": (W, W) for n in "qkvo"})
        s.update({p + "mlp.gate_proj.weight": (F, W), p + "mlp.up_proj.weight": (F, W), p + "mlp.down_proj.weight": (W, F), p + "input_layernorm.weight": (W,),
                  p + "post_attention_layernorm.weight": (W,)})
    s.update({"mm_projector.0.weight": (W, VIS["width"]), "mm_projector.0.bias": (W,), "mm_projector.2.weight": (W, W), "mm_projector.2.bias": (W,)})
    return s


def vision_shapes():
    W, F, p = VIS["width"], VIS["ff"], VIS["patch"]
    s = {"vision.embeddings.class_embedding": (W,), "vision.embeddings.patch_embedding.weight": (W, 3, p, p), "vision.embeddings.position_embedding.weight": (VIS["tokens"] + 1, W),
         "vision.pre_layrnorm.weight": (W,), "vision.pre_layrnorm.bias": (W,)}
    for i in range(VIS["layers"]):
        q = f"vision.encoder.layers.{i}."
        for n, shape in (("self_attn.q_proj", (W, W)), ("self_attn.k_proj", (W, W)), ("self_attn.v_proj", (W, W)), ("self_attn.out_proj", (W, W)), ("mlp.fc1", (F, W)), ("mlp.fc2", (W, F))):
            s[q + n + ".weight"], s[q + n + ".bias"] = shape, shape[:1]
        for n in ("layer_norm1", "layer_norm2"):
            s[q + n + ".weight"], s[q + n + ".bias"] = (W,), (W,)
    return s


def siterax_config(case):
    W, (H, G, D, F) = case["width"], SITERAX[case["width"]]
    layer = {"type": "attention", "mixer": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "mask": {"size": case["window"]} if case["window"] else None,
                                            "rot": {"dims": D, "base": 10000.0}}, "mlp": {"kind": "dense", "ff": F}}
    return {"vocab": VOCAB, "width": W, "layers": [layer] * case["layers"], "norm": {"eps": EPS}, "residual_mult": 0.5, "logit_softcap": 60.0}


def siterax_shapes(case):
    W, (H, G, D, F) = case["width"], SITERAX[case["width"]]
    s = {"embed": (VOCAB, W), "head": (VOCAB, W), "final.norm": (W,)}
    for i in range(case["layers"]):
        p = f"l{i}."
        s.update({p + n: (W,) for n in ("norm1", "norm1b", "norm2", "norm2b")})
        for n, r in (("q", H * D), ("k", G * D), ("v", G * D)):
            s[p + "mix." + n], s[p + f"mix.{n}.b"] = (r, W), (r,)
        s.update({p + "mix.q.norm": (D,), p + "mix.k.norm": (D,), p + "mix.g": (H, W), p + "mix.o": (W, H * D), p + "mlp.gate": (F, W), p + "mlp.up": (F, W), p + "mlp.down": (W, F)})
    return s


def vizosun_config(case):
    """Every fourth layer latent attention, the others the delta rule; every second feed-forward a mixture."""
    W, (H, D, Q, R, F, EF) = case["width"], VIZOSUN[case["width"]]
    layers = []
    for i in range(case["layers"]):
        latent = {"heads": H, "dim": D, "vdim": D, "q_rank": Q, "kv_rank": R, "scale": D ** -0.5, "mask": {"size": case["window"]} if case["window"] else None}
        layers.append({"type": "latent_attention" if i % 4 == 3 else "channel_delta", "mixer": latent if i % 4 == 3 else {"heads": H, "kv_heads": H, "dim": D, "vdim": D, "conv": 4},
                       "mlp": {"kind": "moe", "expert": {"ff": EF}, "router": {"experts": EXPERTS, "top": TOP}} if i % 2 else {"kind": "dense", "ff": F}})
    return {"vocab": VOCAB, "width": W, "layers": layers, "norm": {"eps": EPS}, "embedding": {"bigram": {"buckets": BUCKETS, "mul_prev": MUL[0], "mul_cur": MUL[1]}}, "loop": None}


def vizosun_shapes(case):
    W, (H, D, Q, R, F, EF) = case["width"], VIZOSUN[case["width"]]
    s = {"embed": (VOCAB, W), "bigram": (BUCKETS + 1, W), "final.norm": (W,)}
    for i in range(case["layers"]):
        p, m = f"l{i}.", f"l{i}.mix."
        s[p + "norm1"] = (W,)
        if i % 4 == 3:
            s.update({m + "dq": (Q, W), m + "dq.norm": (Q,), m + "uq": (H * D, Q), m + "dkv": (R, W), m + "dkv.norm": (R,), m + "uk": (H * D, R), m + "uv": (H * D, R)})
        else:
            for n in "qkv":
                s[m + n], s[m + n + ".conv"] = (H * D, W), (H * D, 4)
            s.update({m + "b": (H, W), m + "A_log": (H,), m + "dt_bias": (H * D,), m + "norm": (D,), m + "a1": (RANK, W), m + "a2": (H * D, RANK), m + "g1": (RANK, W), m + "g2": (H * D, RANK)})
        s[m + "o"] = (W, H * D)
        if i % 2:
            s.update({p + "mlp.router": (EXPERTS, W), p + "mlp.router.b": (EXPERTS,)})
            for e in range(EXPERTS):
                q = p + f"mlp.e{e}."
                s.update({q + "gate": (EF, W), q + "up": (EF, W), q + "down": (W, EF)})
        else:
            s.update({p + "mlp.gate": (F, W), p + "mlp.up": (F, W), p + "mlp.down": (W, F)})
    return s


OUTPUTS = ("o_proj.weight", "down_proj.weight", "out_proj.weight", "fc2.weight", ".o", ".down")       # what a sublayer adds to the stream
MARK = 8.0                                                                           # see weight()


def weight(case, seed, name, shape):
    """One tensor, from the seed and its name alone.  A mixture's router follows marks that the stream carries from the embedding on: a trained router tells its tokens
    apart too, and a choice between experts that are level would flip with the last bit of a 16-bit row."""
    dtype, depth = DTYPES[case["dtype"]], case.get("layers", 1)
    vizosun = case["op"].startswith("vizosun")
    if name == "lm_head.weight":
        return head_like(seed, weight(case, seed, "model.embed_tokens.weight", shape))
    if name == "head":
        return head_like(seed, weight(case, seed, "embed", shape))
    if name in ("model.embed_tokens.weight", "embed"):
        t = normal(seed, name, shape, 1.0, dtype)
        if vizosun:                                                                  # the token's own marks
            t[:, :EXPERTS] = MARK * mark_rows(seed, dtype)
        return t
    if name == "bigram":                                                             # the row of a pair holds the token that follows it, louder than the token itself
        t = 1.5 * weight(case, seed, "embed", (VOCAB, shape[1]))[torch.randint(3, VOCAB, shape[:1], generator=seeded(seed, "pairs"), device="cuda")]
        t[:, :EXPERTS] = 0
        return t
    if name.endswith(".router"):
        t = normal(seed, name, shape, 0.02 / shape[1] ** 0.5, dtype)
        t[:, :EXPERTS] += torch.roll(torch.eye(EXPERTS, device="cuda"), int(name.split(".")[0][1:]), 0).to(dtype)
        return t
    if name.endswith(".router.b"):
        return normal(seed, name, shape, 0.01, dtype)
    if name.endswith("A_log"):
        return normal(seed, name, shape, 1.0, dtype, -1.0)
    if name.endswith("dt_bias"):
        return normal(seed, name, shape, 1.0, dtype, -2.0)
    if name.endswith(".conv"):
        return normal(seed, name, shape, 0.5, dtype)
    if len(shape) == 1 and ("norm" in name) and not name.endswith("bias"):
        t = normal(seed, name, shape, 0.1, dtype, 1.0)
        if vizosun and name.endswith("norm1"):
            t[:EXPERTS] = 1
        return t
    if len(shape) == 1:                                                              # biases, the class embedding
        return normal(seed, name, shape, 0.1, dtype)
    if "position_embedding" in name:
        return normal(seed, name, shape, 0.1, dtype)
    if name.endswith(OUTPUTS):
        t = normal(seed, name, shape, (2 * (depth if not name.startswith("vision") else VIS["layers"]) * math.prod(shape[1:])) ** -0.5, dtype)
        if vizosun:
            t[:EXPERTS] = 0
        return t
    return normal(seed, name, shape, math.prod(shape[1:]) ** -0.5, dtype)


def mark_rows(seed, dtype):
    """[VOCAB, EXPERTS] of four larger entries a row, all steps apart."""
    order = torch.rand((VOCAB, EXPERTS), generator=seeded(seed, "marks"), device="cuda").argsort(dim=1)
    level = torch.tensor([1.0, 0.85, 0.7, 0.55] + [-0.3] * (EXPERTS - 4), device="cuda")
    return torch.empty((VOCAB, EXPERTS), device="cuda").scatter_(1, order, level.expand(VOCAB, EXPERTS)).to(dtype)


def pixels(seed, n, dtype):
    """Pictures as the image processor hands them over: smooth, of unit scale."""
    x = torch.empty((n, 3, 42, 42), device="cuda").normal_(generator=seeded(seed, "pixels"))
    fine = torch.empty((n, 3, VIS["size"], VIS["size"]), device="cuda").normal_(0, 0.2, generator=seeded(seed, "grain"))
    return (torch.nn.functional.interpolate(x, size=VIS["size"], mode="bilinear") + fine).to(dtype)


def image_prompt(case, seed):
    ids = prompt(seed, case["rows"], "request")
    at = [min(len(ids), 35 + 7 * i) for i in range(case["images"])]
    for k, a in enumerate(at):
        ids = torch.cat([ids[:a + k], torch.full((1,), IMAGE, device="cuda"), ids[a + k:]])
    return ids


def train_batch(case, seed):
    """(ids, labels, mask) [samples, longest] on the host and the frozen tower's features: every sample an image and a text, the instruction not counted."""
    ns = [max(40, n - VIS["tokens"]) for n in lengths(case, case["rows"])]
    ids, labels, mask = torch.zeros((len(ns), max(ns) + 1), dtype=torch.long), torch.full((len(ns), max(ns) + 1), -100), torch.zeros((len(ns), max(ns) + 1), dtype=torch.bool)
    for i, n in enumerate(ns):
        t = prompt(seed, n, f"sample {i}").cpu()
        ids[i, :n + 1] = torch.cat([t[:20], torch.tensor([IMAGE]), t[20:]])
        labels[i, 33:n + 1] = ids[i, 33:n + 1]
        mask[i, :n + 1] = True
    return ids, labels, mask, normal(seed, "features", (len(ns), VIS["tokens"], VIS["width"]), 1.0, DTYPES[case["dtype"]])


# ---- the calls ----------------------------------------------------------------------------------------------------------------------------------

def llava_config(case, sees=False):
    from llava_mi355x import LlavaConfig
    W, (H, F) = case["width"], LLAVA[case["width"]]
    c = LlavaConfig(hidden_size=W, intermediate_size=F, num_hidden_layers=case.get("layers", 1), num_attention_heads=H, num_key_value_heads=H, vocab_size=VOCAB, rms_norm_eps=EPS,
                    max_position_embeddings=4096, pad_token_id=0, bos_token_id=1, eos_token_id=2)
    c.mm_projector_type, c.mm_hidden_size, c.mm_vision_select_layer, c.mm_vision_select_feature = "mlp2x_gelu", VIS["width"], -2, "patch"
    if sees:
        c.mm_vision_tower = "clip-vit-large-patch14-336"
    return c


def build(case, seed):
    op = case["op"]
    if op.startswith("llava"):
        from llava_mi355x import LlavaLlamaForCausalLM
        from transformers import CLIPVisionConfig
        vision = CLIPVisionConfig(hidden_size=VIS["width"], intermediate_size=VIS["ff"], num_hidden_layers=VIS["layers"], num_attention_heads=VIS["heads"], image_size=VIS["size"],
                                  patch_size=VIS["patch"], layer_norm_eps=EPS, hidden_act="quick_gelu")
        sees = op in ("llava_images", "llava_prompt")
        model = LlavaLlamaForCausalLM(llava_config(case, sees), vision if sees else None, dtype=DTYPES[case["dtype"]], max_position=2560 if op == "llava_prompt" else 2048)
        shapes = llava_shapes(case)
        if sees:
            shapes.update(vision_shapes())
        else:
            shapes = {k: v for k, v in shapes.items() if not k.startswith("mm_projector")}
    elif op.startswith("siterax"):
        from llava_mi355x import SiteraxConfig, SiteraxForCausalLM
        model, shapes = SiteraxForCausalLM(SiteraxConfig.from_dict(siterax_config(case)), dtype=DTYPES[case["dtype"]], max_position=2048), siterax_shapes(case)
    else:
        from llava_mi355x import VizosunConfig, VizosunForCausalLM
        shapes = vizosun_shapes(case)
        model = VizosunForCausalLM(VizosunConfig.from_dict(vizosun_config(case), shapes), dtype=DTYPES[case["dtype"]], max_position=2048)
    for name, shape in shapes.items():
        model.load_tensor(name, weight(case, seed, name, shape))
    model.finalize_weights()
    if model.get_vision_tower() is not None:
        model.get_vision_tower().is_loaded = True
    return model


def prepare(case, seed):
    gc.collect()                                                                     # a model that was dropped gives its gigabytes back to the device now
    op, s = case["op"], {"op": case["op"], "case": case}
    if op == "llava_train":
        from llava_mi355x.train import TrainStep
        shapes = llava_shapes(case)
        s["step"] = TrainStep(llava_config(case), {k: weight(case, seed, k, v) for k, v in shapes.items()}, dtype=DTYPES[case["dtype"]], device="cuda", lr=2e-5, max_positions=2048)
        s["batch"] = train_batch(case, seed)
        return s
    s["model"] = model = build(case, seed)
    if op == "llava_images":
        s["pixels"] = pixels(seed, case["images"], DTYPES[case["dtype"]])
    elif op == "llava_prompt":
        s["ids"], s["pixels"] = image_prompt(case, seed)[None], pixels(seed, case["images"], DTYPES[case["dtype"]]) if case["images"] else None
    elif op == "llava_turn":
        s["ids"] = prompt(seed, case["rows"], "turn")
        s["caches"] = read_prompts(model, [prompt(seed, case["context"], "request 0")])
    elif op.endswith("decode"):
        prompts = [prompt(seed, n, f"request {i}") for i, n in enumerate(lengths(case, case["context"]))]
        s["caches"], s["context"] = read_prompts(model, prompts), [len(p) for p in prompts]
        s["first"] = [int(chain(seed, p[-1:], 1)) for p in prompts]
        s["batch"] = decode_batch(model, len(prompts))
    else:
        s["prompts"] = [prompt(seed, n, f"request {i}") for i, n in enumerate(lengths(case, case["rows"]))]
        s["wants"] = [rows_wanted(len(p)) for p in s["prompts"]]
        s["batch"] = decode_batch(model, len(s["prompts"])) if "tokens" in case else None
    return s


def rows_wanted(n):
    """The rows of a prompt whose logits are asked for: the last one and a few before it."""
    return sorted({n - 1, *range(n // 8, n, max(1, n // 8))})[-8:]


def decode_batch(model, n):
    from llava_mi355x.batching import DecodeBatch
    return DecodeBatch(model, n) if n > 1 else None


def read_prompts(model, prompts):
    """Sequences that hold these prompts."""
    from llava_mi355x._C import check, lib, ptr, stream_handle
    from llava_mi355x.engine_lm import LmxKVCache
    caches = []
    for p in prompts:
        e, c = model.get_model().embed_tokens(p), LmxKVCache(model, 1)
        check(lib.lmx_prefill(model._h, c.seqs[0], ptr(e), len(p), 0, None, 0, 1, stream_handle()), "lmx_prefill")
        torch.cuda.synchronize()
        caches.append(c)
    return caches


def run_decode(model, batch, caches, first, n):
    """n greedy tokens of every sequence behind `first` (None: behind the sequence's own pick): (ids [n, sequences], logits of the last step)."""
    from llava_mi355x._C import check, lib, ptr, stream_handle
    logits = torch.empty((len(caches), model._vocab_cap), dtype=model.logits_dtype, device="cuda")
    if batch is not None:
        ids = batch.step([c.seqs[0] for c in caches], first, n, True, logits)
        return {"ids": torch.tensor(ids), "logits": logits}
    seq, host, got = caches[0].seqs[0], (ctypes.c_int64 * (n + 1))(), ctypes.c_int32(0)
    check(lib.lmx_decode(model._h, seq, first[0] if first else -1, n, ptr(logits), 1, stream_handle()), "lmx_decode")
    check(lib.lmx_seq_read_tokens(seq, host, n + 1, ctypes.byref(got), stream_handle()), "lmx_seq_read_tokens")
    return {"ids": torch.tensor([[t] for t in host[:got.value][-n:]]), "logits": logits}


def run(s):
    op, case = s["op"], s["case"]
    if op == "llava_train":
        ids, labels, mask, features = s["batch"]
        loss, _ = s["step"].step(ids, labels, mask, image_features=features)
        return {"loss": loss, "gradients": s["step"].flat_g, "weights": s["step"].flat_p}
    from llava_mi355x._C import check, lib, ptr, stream_handle
    from llava_mi355x.engine_lm import LmxKVCache
    model = s["model"]
    if op == "llava_images":
        return model.encode_images(s["pixels"])
    if op == "llava_prompt":
        if s["pixels"] is not None:
            embeds = model.prepare_inputs_labels_for_multimodal(s["ids"], None, None, None, None, s["pixels"])[4][0]
        else:
            embeds = model.get_model().embed_tokens(s["ids"])[0]
        cache, logits = LmxKVCache(model, 1), torch.empty((1, model._vocab_cap), dtype=model.logits_dtype, device="cuda")
        check(lib.lmx_prefill(model._h, cache.seqs[0], ptr(embeds), embeds.shape[0], 0, ptr(logits), 0, 1, stream_handle()), "lmx_prefill")
        cache.close()
        return logits
    if op == "llava_turn":
        seq, logits = s["caches"][0].seqs[0], torch.empty((1, model._vocab_cap), dtype=model.logits_dtype, device="cuda")
        check(lib.lmx_seq_truncate(seq, case["context"], stream_handle()), "lmx_seq_truncate")
        embeds = model.get_model().embed_tokens(s["ids"])
        check(lib.lmx_prefill(model._h, seq, ptr(embeds), embeds.shape[0], 0, ptr(logits), 0, 1, stream_handle()), "lmx_prefill")
        return logits
    if op.endswith("decode"):
        for c, n in zip(s["caches"], s["context"]):
            check(lib.lmx_seq_truncate(c.seqs[0], n, stream_handle()), "lmx_seq_truncate")
        return run_decode(model, s["batch"], s["caches"], s["first"], case["tokens"])
    caches = [LmxKVCache(model, 1) for _ in s["prompts"]]
    embeds = model.get_model().embed_tokens(torch.cat(s["prompts"])).split([len(p) for p in s["prompts"]])
    if op.endswith("prompt"):
        out = {"logits": model.prefill_logits(caches, embeds, s["wants"])}
    else:
        n = len(caches)
        check(lib.lmx_prefill_batch(model._h, (ctypes.c_void_p * n)(*[c.seqs[0].value for c in caches]), n, (ctypes.c_void_p * n)(*[e.data_ptr() for e in embeds]),
                                    (ctypes.c_int32 * n)(*[e.shape[0] for e in embeds]), 0, 1, stream_handle()), "lmx_prefill_batch")
        out = run_decode(model, s["batch"], caches, None, case["tokens"])
    for c in caches:
        c.close()
    return out


# ---- the same results in 64 bits ------------------------------------------------------------------------------------------------------------------

class Weights:
    """w[name]: the tensor in 64 bits, made when it is asked for."""

    def __init__(self, case, seed, shapes):
        self.case, self.seed, self.shapes = case, seed, shapes

    def __getitem__(self, name):
        return weight(self.case, self.seed, name, self.shapes[name]).double()


def rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def silu(z):
    return z * torch.sigmoid(z)


def rotate(x, base=10000.0):
    """Rotary positions 0 .. T-1 of x [B, T, heads, D], dimension i with i + D / 2."""
    T, D = x.shape[1], x.shape[3]
    ang = torch.arange(T, dtype=torch.float64, device="cuda")[:, None] * base ** (-torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def attend(q, k, v, scale, window=0, sink=False, causal=True):
    """softmax(scale q k^T) v over [B, T, heads, D]; a sink is one more key of score 0 without a value."""
    B, T, H, _ = q.shape
    rep = H // k.shape[2]
    out = torch.empty((B, T, H, v.shape[3]), dtype=torch.float64, device="cuda")
    i = torch.arange(T, device="cuda")
    hidden = (i[None] > i[:, None]) | ((i[:, None] - i[None] >= window) if window else False)
    for b in range(B):
        for h in range(H):
            s = q[b, :, h] @ k[b, :, h // rep].T.contiguous() * scale
            if causal:
                s = s.masked_fill(hidden, -math.inf)
            if sink:
                s = torch.cat([s, torch.zeros((T, 1), dtype=s.dtype, device="cuda")], 1)
            out[b, :, h] = torch.softmax(s, -1)[:, :T] @ v[b, :, h // rep]
    return out.reshape(B, T, -1)


def exact_images(case, seed, x):
    """[n * tokens, width]: the tower's layer -2 without its class row, through the projector."""
    shapes = {**vision_shapes(), **llava_shapes({**case, "layers": 0})}
    w, W, n, H, norm = Weights(case, seed, shapes), VIS["width"], x.shape[0], VIS["heads"], torch.nn.functional.layer_norm
    p = "vision.embeddings."
    rows = torch.nn.functional.unfold(x.double(), VIS["patch"], stride=VIS["patch"]).transpose(1, 2) @ w[p + "patch_embedding.weight"].reshape(W, -1).T
    h = torch.cat([w[p + "class_embedding"].expand(n, 1, W), rows], 1) + w[p + "position_embedding.weight"]
    h = norm(h, (W,), w["vision.pre_layrnorm.weight"], w["vision.pre_layrnorm.bias"], EPS)
    for i in range(VIS["run"]):
        p = f"vision.encoder.layers.{i}."
        lin = lambda y, m: y @ w[p + m + ".weight"].T + w[p + m + ".bias"]  # noqa: E731
        y = norm(h, (W,), w[p + "layer_norm1.weight"], w[p + "layer_norm1.bias"], EPS)
        q, k, v = (lin(y, f"self_attn.{m}_proj").view(n, -1, H, W // H) for m in "qkv")
        h = h + lin(attend(q, k, v, (W // H) ** -0.5, causal=False), "self_attn.out_proj")
        y = lin(norm(h, (W,), w[p + "layer_norm2.weight"], w[p + "layer_norm2.bias"], EPS), "mlp.fc1")
        h = h + lin(y * torch.sigmoid(1.702 * y), "mlp.fc2")
    return project(h[:, 1:].reshape(-1, W), w)


def project(x, w):
    x = torch.nn.functional.gelu(x @ w["mm_projector.0.weight"].T + w["mm_projector.0.bias"])
    return x @ w["mm_projector.2.weight"].T + w["mm_projector.2.bias"]


def llava_layer(x, w, i, H):
    p, (B, T, W) = f"model.layers.{i}.", x.shape
    h = rms(x, w[p + "input_layernorm.weight"])
    q, k, v = ((h @ w[p + f"self_attn.{n}_proj.weight"].T).view(B, T, H, W // H) for n in "qkv")
    x = x + attend(rotate(q), rotate(k), v, (W // H) ** -0.5) @ w[p + "self_attn.o_proj.weight"].T
    h = rms(x, w[p + "post_attention_layernorm.weight"])
    return x + (silu(h @ w[p + "mlp.gate_proj.weight"].T) * (h @ w[p + "mlp.up_proj.weight"].T)) @ w[p + "mlp.down_proj.weight"].T


def llava_rows(case, seed, x):
    """The stream behind the last layer and its norm, x [B, T, width]."""
    w = Weights(case, seed, llava_shapes(case))
    for i in range(case["layers"]):
        x = llava_layer(x, w, i, LLAVA[case["width"]][0])
    return rms(x, w["model.norm.weight"])


def siterax_rows(case, seed, ids):
    W, (H, G, D, _) = case["width"], SITERAX[case["width"]]
    w = Weights(case, seed, siterax_shapes(case))
    x = w["embed"][ids]
    B, T, _ = x.shape
    for i in range(case["layers"]):
        p = f"l{i}."
        m = p + "mix."
        h = rms(x, w[p + "norm1"])
        q, k, v = ((h @ w[m + n].T + w[m + n + ".b"]).view(B, T, -1, D) for n in "qkv")
        o = attend(rotate(rms(q, w[m + "q.norm"])), rotate(rms(k, w[m + "k.norm"])), v, D ** -0.5, case["window"], sink=True).view(B, T, H, D)
        o = (o * torch.sigmoid(h @ w[m + "g"].T)[..., None]).reshape(B, T, -1) @ w[m + "o"].T
        x = x + 0.5 * rms(o, w[p + "norm1b"])
        h = rms(x, w[p + "norm2"])
        x = x + 0.5 * rms((silu(h @ w[p + "mlp.gate"].T) * (h @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T, w[p + "norm2b"])
    return rms(x, w["final.norm"])


def bigram_bucket(prev, cur):
    return (prev * MUL[0] + cur * MUL[1]) % BUCKETS


def delta_mixer(h, w, m, H, D):
    B, T, _ = h.shape

    def conv(n):
        y = torch.nn.functional.pad(h @ w[m + n].T, (0, 0, 3, 0))
        t = w[m + n + ".conv"]
        return silu(sum(y[:, j:j + T] * t[:, j] for j in range(4))).view(B, T, H, D)

    def unit(y):
        return y * torch.rsqrt((y * y).sum(-1, keepdim=True) + 1e-6)

    q, k, v = unit(conv("q")) * D ** -0.5, unit(conv("k")), conv("v")
    z = torch.nn.functional.softplus(h @ w[m + "a1"].T @ w[m + "a2"].T + w[m + "dt_bias"]).view(B, T, H, D)
    g, beta = torch.exp(-torch.exp(w[m + "A_log"])[:, None] * z), torch.sigmoid(h @ w[m + "b"].T)
    S, out = torch.zeros((B, H, D, D), dtype=torch.float64, device="cuda"), torch.empty_like(v)
    for t in range(T):
        S = S * g[:, t, :, :, None]
        u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
        S = S + k[:, t, :, :, None] * u[:, :, None]
        out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    gate = torch.sigmoid(h @ w[m + "g1"].T @ w[m + "g2"].T).view(B, T, H, D)
    return (rms(out, w[m + "norm"]) * gate).reshape(B, T, -1) @ w[m + "o"].T


def latent_mixer(h, w, m, H, D, window):
    B, T, _ = h.shape
    c = rms(h @ w[m + "dkv"].T, w[m + "dkv.norm"])
    q, k, v = ((y @ w[m + n].T).view(B, T, H, D) for y, n in ((rms(h @ w[m + "dq"].T, w[m + "dq.norm"]), "uq"), (c, "uk"), (c, "uv")))
    return attend(q, k, v, D ** -0.5, window) @ w[m + "o"].T


def vizosun_rows(case, seed, ids):
    W, (H, D, _, _, _, _) = case["width"], VIZOSUN[case["width"]]
    w = Weights(case, seed, vizosun_shapes(case))
    pair = torch.cat([torch.full_like(ids[:, :1], BUCKETS), bigram_bucket(ids[:, :-1], ids[:, 1:])], 1)
    x = w["embed"][ids] + w["bigram"][pair]
    for i in range(case["layers"]):
        p = f"l{i}."
        h = rms(x, w[p + "norm1"])
        y = latent_mixer(h, w, p + "mix.", H, D, case["window"]) if i % 4 == 3 else delta_mixer(h, w, p + "mix.", H, D)
        if i % 2:
            f = h.reshape(-1, W)
            best, at = (f @ w[p + "mlp.router"].T + w[p + "mlp.router.b"]).topk(TOP, dim=-1)
            best, z = torch.softmax(best, -1), torch.zeros_like(f)
            for e in range(EXPERTS):
                r, j = (at == e).nonzero(as_tuple=True)
                q = p + f"mlp.e{e}."
                z[r] += best[r, j, None] * ((silu(f[r] @ w[q + "gate"].T) * (f[r] @ w[q + "up"].T)) @ w[q + "down"].T)
            y = y + z.view_as(h)
        else:
            y = y + (torch.relu(h @ w[p + "mlp.gate"].T) * (h @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T
        x = x + y
    return rms(x, w["final.norm"])


def padded(rows):
    """[B, longest]: what stands behind a request's end does not reach back."""
    return torch.nn.utils.rnn.pad_sequence(rows, batch_first=True)


def exact(case, seed):
    op = case["op"]
    if op == "llava_images":
        return exact_images(case, seed, pixels(seed, case["images"], DTYPES[case["dtype"]])).view(case["images"], VIS["tokens"], case["width"])
    if op == "llava_train":
        return exact_train(case, seed)
    with torch.no_grad():
        if op == "llava_prompt":
            ids = image_prompt(case, seed)
            x = weight(case, seed, "model.embed_tokens.weight", (VOCAB, case["width"])).double()[ids.clamp(min=0)]
            if case["images"]:
                feats = exact_images(case, seed, pixels(seed, case["images"], DTYPES[case["dtype"]])).split(VIS["tokens"])
                parts, at = [], 0
                for f, a in zip(feats, (ids == IMAGE).nonzero()[:, 0].tolist()):
                    parts += [x[at:a], f]
                    at = a + 1
                x = torch.cat(parts + [x[at:]])
            last = llava_rows(case, seed, x[None])[:, -1]
            return last @ weight(case, seed, "lm_head.weight", (VOCAB, case["width"])).double().T
        if op == "llava_turn":
            rows = [torch.cat([prompt(seed, case["context"], "request 0"), prompt(seed, case["rows"], "turn")])]
        elif op.endswith("decode"):
            rows = [prompt(seed, n, f"request {i}") for i, n in enumerate(lengths(case, case["context"]))]
            picks = chain(seed, torch.stack([r[-1] for r in rows]), case["tokens"] + 1)
            rows, ids = [torch.cat([r, picks[:-1, i]]) for i, r in enumerate(rows)], picks[1:]
        else:
            rows = [prompt(seed, n, f"request {i}") for i, n in enumerate(lengths(case, case["rows"]))]
            if "tokens" in case:
                table = torch.randint(3, VOCAB, (BUCKETS + 1,), generator=seeded(seed, "pairs"), device="cuda")
                for _ in range(case["tokens"]):
                    rows = [torch.cat([r, table[bigram_bucket(r[-2:-1], r[-1:])]]) for r in rows]
                ids = torch.stack([torch.cat([r[-case["tokens"]:][1:], table[bigram_bucket(r[-2:-1], r[-1:])]]) for r in rows], 1)
        name, width = ("lm_head.weight" if op.startswith("llava") else "head" if op.startswith("siterax") else "embed"), case["width"]
        if op.startswith("llava"):
            embed = weight(case, seed, "model.embed_tokens.weight", (VOCAB, width)).double()
            h = llava_rows(case, seed, embed[padded(rows)])
        else:
            h = (siterax_rows if op.startswith("siterax") else vizosun_rows)(case, seed, padded(rows))
        at = [rows_wanted(len(r)) if op in ("siterax_prompt", "vizosun_prompt") else [len(r) - 1] for r in rows]
        z = torch.cat([h[i, a] for i, a in enumerate(at)]) @ weight(case, seed, name, (VOCAB, width)).double().T
        if op.startswith("siterax"):
            z = 60.0 * torch.tanh(z / 60.0)
        return {"ids": ids, "logits": z} if "tokens" in case else z if op == "llava_turn" else {"logits": z}


def exact_train(case, seed):
    """Loss, gradients and stepped weights, flat in the order in which the gradients are done."""
    shapes, W, H = llava_shapes(case), case["width"], LLAVA[case["width"]][0]
    w = {k: weight(case, seed, k, v).double().requires_grad_(True) for k, v in shapes.items()}
    ids, labels, mask, features = train_batch(case, seed)
    loss, counted = 0.0, int((labels[:, 1:] != -100).sum())
    for i in range(ids.shape[0]):
        t, l = ids[i][mask[i]], labels[i][mask[i]]
        a = int((t == IMAGE).nonzero())
        x = torch.cat([w["model.embed_tokens.weight"][t[:a].cuda()], project(features[i].double(), w), w["model.embed_tokens.weight"][t[a + 1:].cuda()]])[None]
        l = torch.cat([l[:a], torch.full((VIS["tokens"],), -100), l[a + 1:]]).cuda()
        for k in range(case["layers"]):
            x = llava_layer(x, w, k, H)
        z = rms(x, w["model.norm.weight"])[0] @ w["lm_head.weight"].T
        part = torch.nn.functional.cross_entropy(z[:-1], l[1:], ignore_index=-100, reduction="sum") / counted
        part.backward()
        loss += part.detach()
    order = ["lm_head.weight", "model.norm.weight"]
    for k in reversed(range(case["layers"])):
        p = f"model.layers.{k}."
        order += [p + n for n in ("mlp.down_proj.weight", "mlp.gate_proj.weight", "mlp.up_proj.weight", "post_attention_layernorm.weight", "self_attn.o_proj.weight",
                                  "self_attn.q_proj.weight", "self_attn.k_proj.weight", "self_attn.v_proj.weight", "input_layernorm.weight")]
    order += ["mm_projector.2.bias", "mm_projector.2.weight", "mm_projector.0.bias", "mm_projector.0.weight", "model.embed_tokens.weight"]
    g = torch.cat([w[n].grad.reshape(-1) for n in order])
    p = torch.cat([w[n].detach().reshape(-1) for n in order])
    clipped = g * (1.0 / (g.norm() + 1e-6)).clamp(max=1.0)
    return {"loss": loss, "gradients": g, "weights": p - 2e-5 * clipped / (clipped.abs() + 1e-8)}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------------------------------

def work(case):
    op, W = case["op"], case["width"]
    if op.startswith("llava"):
        H, F = LLAVA[W]
        layer, heads, seen_flops, kv_bytes, active = 4 * W * W + 3 * W * F, H, 4 * W, 4 * W, 1.0
    elif op.startswith("siterax"):
        H, G, D, F = SITERAX[W]
        layer, seen_flops, kv_bytes, active = W * D * (2 * H + 2 * G) + 3 * W * F, 4 * H * D, 4 * G * D, 1.0
    if op == "llava_images":
        v, n = vision_work(), case["images"]
        proj = VIS["width"] * W + W * W
        return {"bytes": 2 * (v["params"] + proj) + n * (6 * VIS["size"] ** 2 + 2 * VIS["tokens"] * W), "flops": n * (v["flops"] + 2 * VIS["tokens"] * proj)}
    if op == "llava_train":
        ns = [max(40, n - VIS["tokens"]) + VIS["tokens"] for n in lengths(case, case["rows"])]
        params = case["layers"] * layer + VOCAB * W
        return {"bytes": (params + VOCAB * W) * (2 + 2 + 2 + 24), "flops": sum(6 * params * n + case["layers"] * 3 * seen_flops * n * n / 2 for n in ns)}
    if op == "llava_prompt":
        n = case["rows"] + VIS["tokens"] * case["images"]
        out = {"bytes": 2 * (case["layers"] * layer + VOCAB * W) + case["layers"] * kv_bytes * n, "flops": n * case["layers"] * (2 * layer + seen_flops * n / 2) + 2 * VOCAB * W}
        if case["images"]:
            v = work({"op": "llava_images", "width": W, "images": case["images"]})
            out = {k: out[k] + v[k] for k in out}
        return out
    if op == "llava_turn":
        n, c = case["rows"], case["context"]
        return {"bytes": 2 * (case["layers"] * layer + VOCAB * W) + case["layers"] * kv_bytes * (2 * n + c), "flops": n * case["layers"] * (2 * layer + seen_flops * (c + n / 2)) + 2 * VOCAB * W}
    L, n = case["layers"], case["requests"]
    if op.startswith("vizosun"):
        return vizosun_work(case)
    window = case.get("window", 0) or 1 << 30
    if op.endswith("prompt"):
        ns = lengths(case, case["rows"])
        seen = sum(sum(min(i + 1, window) for i in range(m)) for m in ns)
        return {"bytes": 2 * (L * layer + VOCAB * W) + L * kv_bytes * sum(ns), "flops": 2 * L * layer * sum(ns) + L * seen_flops * seen + 16 * n * VOCAB * W}
    keys = sum(min(m + case["tokens"] / 2, window) for m in lengths(case, case["context"]))
    t = case["tokens"]
    return {"bytes": t * (2 * (L * layer + VOCAB * W) + L * kv_bytes * keys), "flops": t * (2 * (L * layer + VOCAB * W) * n + L * seen_flops * keys)}


def vision_work():
    W, F, T = VIS["width"], VIS["ff"], VIS["tokens"] + 1
    params = VIS["run"] * (4 * W * W + 2 * W * F) + 3 * VIS["patch"] ** 2 * W
    return {"params": params, "flops": 2 * T * params + VIS["run"] * 4 * T * T * W}


def vizosun_work(case):
    W, (H, D, Q, R, F, EF) = case["width"], VIZOSUN[case["width"]]
    L, n, hd = case["layers"], case["requests"], H * D
    ns = lengths(case, case["rows"])
    latent, delta = L // 4, L - L // 4
    mixed, plain = L // 2, L - L // 2
    mixer = latent * (W * (Q + R) + hd * (Q + 2 * R) + W * hd) + delta * (4 * W * hd + 2 * RANK * (W + hd))
    per_row = mixer + plain * 3 * W * F + mixed * 3 * W * EF * TOP                                        # weights a row is multiplied with
    state = delta * 7 * hd * D

    def once(rows):                                                                                       # weights that so many rows touch at all
        return 2 * (mixer + plain * 3 * W * F + mixed * 3 * W * EF * EXPERTS * (1 - (1 - TOP / EXPERTS) ** rows) + VOCAB * W)

    rows = sum(ns)
    out = {"bytes": once(rows) + delta * 8 * hd * D * n, "flops": rows * (2 * per_row + state) + latent * 2 * hd * sum(m * min(m, case["window"] or m) for m in ns) + 16 * n * VOCAB * W}
    if "tokens" in case:
        t = case["tokens"]
        out["bytes"] += t * (once(n) + delta * 8 * hd * D * n + latent * 2 * R * sum(ns))
        out["flops"] += t * n * (2 * per_row + state + 2 * VOCAB * W)
    return out


def tolerance(case):
    """Four times the distance from 64 bits that was measured; ids are the same ones."""
    op, deep = case["op"], case.get("layers", 0) > 8
    if op == "llava_train":
        rel = 0.015
    elif op.startswith("llava"):
        rel = 0.03 if deep and case["dtype"] == "bf16" else 0.024
        if op == "llava_images":
            rel = 0.03
        if case["dtype"] == "f16":
            rel = 0.006
    else:
        rel = 0.02 if op.startswith("siterax") else 0.0075
    return {"rel": rel, "differ": 0.0}
