"""Prompt attention on both query-block forms (64 rows where 128 would leave CUs idle, 128 where the blocks fill the chip) against the same attention in float64: sizes around the tiles and
blocks of each, slices of the window, scales of either sign and zero."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16}


def dense(q, k, vt, heads, scale, pos0, causal, window=0, sink=False):
    """(softmax(scale q k^T) v, the same of |v|) in float64."""
    T, D, kv = q.shape[0], k.shape[2], k.shape[1]
    q = q.double().view(T, heads, D).transpose(0, 1)
    rep = heads // k.shape[0]
    k, v = k.double().repeat_interleave(rep, 0), vt.double().repeat_interleave(rep, 0).transpose(1, 2).contiguous()
    s = torch.stack([q[h] @ k[h].T.contiguous() for h in range(heads)]) * scale
    i, j = torch.arange(T, device="cuda")[:, None] + pos0, torch.arange(kv, device="cuda")[None]
    if causal:
        s = s.masked_fill((j > i) | ((i - j >= window) if window else False), -math.inf)
    if sink:
        s = torch.cat([s, torch.zeros_like(s[:, :, :1])], 2)
    p = torch.softmax(s, -1)[:, :, :kv]
    return [torch.stack([p[h] @ x[h] for h in range(heads)]).transpose(0, 1).reshape(T, heads * D) for x in (v, v.abs())]


def problem(dt, T, kv, heads, kv_heads, D):
    g = torch.Generator(device="cuda").manual_seed(T * 1009 + kv)
    s_max = (kv + 63) // 64 * 64
    rnd = lambda *shape: torch.empty(shape, dtype=dt, device="cuda").normal_(generator=g)  # noqa: E731
    q, k, vt = rnd(T, heads * D), rnd(kv_heads, s_max, D), rnd(kv_heads, D, s_max)
    vt[:, :, kv:] = 0                                                        # as the caches' writers leave what lies behind the last key
    return q, k, vt


def near(got, want, absolute, dt):
    # every probability is rounded once, the output once more: 8 significant bits (bf16) or 11 (f16) are at most 2^-8 or 2^-11 off, relative; 1e-5 for the fp32 exponentials and sums
    half = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    bound = absolute * (half + 1e-5) + want.abs() * half + 1e-6
    assert bool(((got.double() - want).abs() <= 1.01 * bound).all()), ((got.double() - want).abs() / bound).max().item()


@pytest.mark.parametrize("name", DT)
@pytest.mark.parametrize("T,ctx,heads,kv_heads", [
    (1, 0, 4, 4), (31, 0, 4, 2), (32, 1, 4, 4), (33, 31, 4, 1), (63, 0, 8, 8), (64, 0, 8, 2), (65, 63, 4, 4), (97, 32, 4, 4), (129, 0, 4, 2), (191, 66, 8, 2), (320, 5, 4, 4),      # 64-row blocks
    (128, 130, 256, 8), (127, 64, 256, 8), (100, 1, 256, 4), (256, 700, 128, 4), (130, 400, 128, 4),                                                                                   # 128-row blocks
])
def test_causal_against_float64(cuda, name, T, ctx, heads, kv_heads):
    from llava_mi355x import ops
    dt, D = DT[name], 128
    q, k, vt = problem(dt, T, T + ctx, heads, kv_heads, D)
    got = ops.flash_attn(q, k, vt, T, T + ctx, ctx, heads, kv_heads, D, True)
    near(got, *dense(q, k[:, :T + ctx], vt[:, :, :T + ctx], heads, D ** -0.5, ctx, True), dt)


@pytest.mark.parametrize("T,kv,heads,D", [(65, 65, 4, 64), (128, 191, 4, 64), (5, 33, 4, 128), (128, 95, 256, 128), (77, 320, 256, 128)])
def test_without_a_causal_limit(cuda, T, kv, heads, D):
    from llava_mi355x import ops
    q, k, vt = problem(torch.float16, T, kv, heads, heads // 4, D)
    near(ops.flash_attn(q, k, vt, T, kv, 0, heads, heads // 4, D, False), *dense(q, k[:, :kv], vt[:, :, :kv], heads, D ** -0.5, 0, False), torch.float16)


@pytest.mark.parametrize("scale", [128 ** -0.5, -0.05, 0.0])
@pytest.mark.parametrize("T,ctx,heads,window", [(70, 200, 4, 33), (130, 0, 4, 64), (200, 31, 4, 0), (128, 500, 256, 100), (129, 380, 128, 0)])
def test_windows_and_scales(cuda, scale, T, ctx, heads, window):
    from llava_mi355x import ops
    q, k, vt = problem(torch.bfloat16, T, T + ctx, heads, heads // 4, 128)
    got = ops.window_attn(q, k, vt, ctx, heads, heads // 4, scale, window=window, sink=True)
    near(got, *dense(q, k[:, :T + ctx], vt[:, :, :T + ctx], heads, scale, ctx, True, window, True), torch.bfloat16)


def test_log_sum_exp_of_both_forms(cuda):
    from llava_mi355x import ops
    for T, ctx, heads in ((97, 0, 4), (128, 300, 256)):
        q, k, vt = problem(torch.bfloat16, T, T + ctx, heads, 4, 128)
        lse = torch.empty((heads, T), device="cuda")
        ops.flash_attn(q, k, vt, T, T + ctx, ctx, heads, 4, 128, True, lse=lse)
        s = torch.stack([q.double().view(T, heads, 128)[:, h] @ k[h * 4 // heads, :T + ctx].double().T.contiguous() for h in range(heads)]) * 128 ** -0.5
        i, j = torch.arange(T, device="cuda")[:, None] + ctx, torch.arange(T + ctx, device="cuda")[None]
        want = torch.logsumexp(s.masked_fill(j > i, -math.inf), -1) / math.log(2)
        assert (lse.double() - want).abs().max().item() < 2e-5 * want.abs().max().item()      # fp32: scores of 128 products, sums of up to 428 exponentials


@pytest.mark.parametrize("name", DT)
@pytest.mark.parametrize("lens,pos0,heads,D,window,rows", [
    ([1, 65, 200, 31], [0, 63, 5, 300], 4, 128, 0, 64), ([40, 129, 64, 97], [10, 0, 190, 1], 8, 128, 33, 64), ([5, 130, 64], [70, 0, 1], 4, 64, 0, 128), ([63, 1], [2, 500], 4, 64, 100, 128),
    ([128, 128], [700, 640], 256, 128, 0, 128), ([3, 256, 255], [8, 500, 450], 128, 128, 0, 128), ([128, 128], [1300, 1200], 256, 128, 1024, 128),
])
def test_rows_of_several_sequences(cuda, name, lens, pos0, heads, D, window, rows):
    """Both forms, sequences out of order and of unlike length, gates and a sink."""
    from llava_mi355x import ops
    dt, kv_heads = DT[name], heads // 4
    assert ops.flash_segs_plan(lens, pos0, heads, D, window)[0] == rows
    s_max = max((p + n + 63) // 64 * 64 for p, n in zip(pos0, lens))
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + heads)
    rnd = lambda *shape: torch.empty(shape, dtype=dt, device="cuda").normal_(generator=g)  # noqa: E731
    qkv = rnd(sum(lens), heads * D + (heads + 7) // 8 * 8)
    ks, vts = [rnd(kv_heads, s_max, D) for _ in lens], [rnd(kv_heads, D, s_max) for _ in lens]
    for vt, p, n in zip(vts, pos0, lens):
        vt[:, :, p + n:] = 0
    got = ops.window_attn_segs(qkv, lens, pos0, ks, vts, heads, kv_heads, D ** -0.5, window=window, sink=True, gate_off=heads * D)
    at = 0
    for n, p, k, vt in zip(lens, pos0, ks, vts):
        r = slice(at, at + n)
        gate = torch.sigmoid(qkv[r, heads * D:heads * D + heads].double()).repeat_interleave(D, 1)
        want, absolute = dense(qkv[r, :heads * D].contiguous(), k[:, :p + n], vt[:, :, :p + n], heads, D ** -0.5, p, True, window, True)
        near(got[r], want * gate, absolute * gate, dt)
        at += n
