"""One new token of several sequences, all query heads of a kv head in one workgroup (csrc/stack_ops.hip: decode_win_group_kernel): group sizes up to the tile's 16 columns and
one past it, positions at the borders of a wave's 32 and a chunk's 128 keys, windows that start inside either, splits without a chunk; against float64 and against the
same sequence on its own (the one-head-per-workgroup kernel)."""
import math

import pytest
import torch

from test_siterax_ops_gpu import DT, TOL, _attn_oracle, _err, _pad, _qkv, _table
from oracle import siterax_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("H,G,D,dim", [(16, 1, 128, 128), (17, 1, 64, 64), (8, 4, 128, 96), (15, 3, 64, 40)])
@pytest.mark.parametrize("window", [0, 33, 160])
@pytest.mark.parametrize("n_split", [1, 3, 9])
def test_groups(cuda, dt, H, G, D, dim, window, n_split):
    from llava_mi355x import ops
    s_max, eps, scale, rot = 1280, 1e-5, 0.9 * dim ** -0.5, dim // 2
    positions = [31, 32, 33, 128, 159, 161, 1279]
    stride, n = (H + 2 * G) * D + 64, len(positions)
    row, q, k, v = _qkv(n, H, G, D, dim, dim, stride, dt, 3)
    g = torch.Generator().manual_seed(9)
    nw = _pad((1 + 0.3 * torch.randn(dim, generator=g)).to(DT[dt]), D)
    r = {"dims": rot, "base": 500.0, "scaling": {"factor": 1.5}}
    tab = _table(r, s_max).to(cuda)

    def caches():
        c = torch.Generator().manual_seed(21)
        ks, vs, old = [], [], []
        for p in positions:
            kk, vv = torch.randn(s_max, G, dim, generator=c).to(DT[dt]), torch.randn(s_max, G, dim, generator=c).to(DT[dt])
            kc, vt = _pad(kk, D).transpose(0, 1).contiguous(), _pad(vv, D).permute(1, 2, 0).contiguous()
            kc[:, p:], vt[:, :, p:] = float("nan"), float("inf")
            if window and p >= window:
                vt[:, :, :p - window + 1] = float("nan")
            ks.append(kc.to(cuda)); vs.append(vt.to(cuda)); old.append((kk[:p].double(), vv[:p].double()))
        return ks, vs, old
    words = [torch.tensor([p], dtype=torch.int32, device=cuda) for p in positions]
    ks, vs, old = caches()
    args = (tab, H, G, dim, rot, scale, eps, nw.to(cuda), nw.to(cuda), window, True, -1, n_split)
    got = ops.decode_win(row.to(cuda), ks, vs, words, *args).reshape(n, H, D)
    k1, v1, _ = caches()
    rd = lambda x: x.to(DT[dt]).double()
    for i, p in enumerate(positions):
        pos = torch.tensor([p])
        qi, ki = (rd(O.rotate(O.rms_norm(x[i:i + 1], nw[:dim].double(), eps), pos, r)) for x in (q, k))
        want = _attn_oracle(qi, torch.cat([old[i][0], ki]), torch.cat([old[i][1], v[i:i + 1]]), p, window, True, None, scale)
        assert _err(got[i:i + 1, :, :dim], want) < TOL[dt], p
        alone = ops.decode_win(row[i:i + 1].to(cuda), k1[i:i + 1], v1[i:i + 1], words[i:i + 1], *args).reshape(H, D)
        assert _err(got[i], alone.double().cpu()) < TOL[dt] and torch.equal(ks[i][:, p], k1[i][:, p]) and torch.equal(vs[i][:, :, p], v1[i][:, :, p])


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("n_split", [1, 3])
def test_small_probabilities(cuda, dt, n_split):
    """One key of weight 1 whose value is 0 and a tail of 1000 keys of weights 2^-22 .. 2^-27: the output is the tail's alone, to the bits of fp32 weights.  Bound: the output's
    rounding, the fp32 sum's 1000 terms, a score's rounding (27 x 2^-23 in the exponent)."""
    from llava_mi355x import ops
    H, G, D, n, tail = 4, 1, 64, 2, 1000
    T = DT[dt]
    g = torch.Generator().manual_seed(4)
    row = torch.zeros(n, (H + 2 * G) * D)
    row[:, [h * D for h in range(H)]] = 1
    row[:, H * D] = -100                                                         # the new key: out of sight
    k, v = torch.zeros(n, 1, tail + 128 - tail % 128, D), torch.zeros(n, 1, D, tail + 128 - tail % 128)
    k[:, 0, 1:tail + 1, 0] = -(22 + 5 * torch.rand(n, tail, generator=g))
    v[:, 0, :, 1:tail + 1] = 1024 * (0.5 + 0.5 * torch.rand(n, D, tail, generator=g))
    k, v = k.to(T), v.to(T)
    words = [torch.tensor([tail + 1], dtype=torch.int32, device=cuda) for _ in range(n)]
    got = ops.decode_win(row.to(T).to(cuda), [c.to(cuda) for c in k], [c.to(cuda) for c in v], words, None, H, G, D, 0, math.log(2.0), 1e-5, sink=False, n_split=n_split)
    p = torch.exp2(k[:, 0, :tail + 1, 0].double())
    want = (v[:, 0, :, :tail + 1].double() @ p.unsqueeze(2)).squeeze(2) / p.sum(1, keepdim=True)
    bound = (2.0 ** -8 if dt == "bf16" else 2.0 ** -11) + tail * 2.0 ** -24 + 27 * 2.0 ** -23
    assert ((got.double().cpu().view(n, H, D) - want[:, None]).abs() <= bound * want[:, None]).all()
