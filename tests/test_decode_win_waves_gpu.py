"""The grouped windowed decode with eight waves a workgroup (csrc/stack_ops.hip: decode_win_group_kernel): windows that start inside a piece and reach past one round of the eight waves'
pieces, splits that hand over to each other, splits and waves without a piece; against float64 and against the same sequence on its own (one head a workgroup)."""
import math

import pytest
import torch

from test_siterax_ops_gpu import DT, TOL, _attn_oracle, _err, _pad, _qkv, _table
from oracle import siterax_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("H,G,D,dim", [(16, 1, 128, 128), (8, 4, 128, 96), (15, 3, 64, 40)])
@pytest.mark.parametrize("window", [0, 33, 160, 600, 1024])
@pytest.mark.parametrize("n_split", [1, 2, 3, 9])
@pytest.mark.parametrize("waves", [4, 8])
def test_waves(cuda, dt, H, G, D, dim, window, n_split, waves):
    from llava_mi355x import ops
    s_max, eps, scale, rot = 1280, 1e-5, 0.9 * dim ** -0.5, dim // 2
    positions = [0, 63, 64, 511, 512, 513, 1100, 1279]
    stride, n = (H + 2 * G) * D + 64, len(positions)
    row, q, k, v = _qkv(n, H, G, D, dim, dim, stride, dt, 3)
    g = torch.Generator().manual_seed(9)
    nw = _pad((1 + 0.3 * torch.randn(dim, generator=g)).to(DT[dt]), D)
    r = {"dims": rot, "base": 500.0, "scaling": {"factor": 1.5}}
    tab = _table(r, s_max).to(cuda)
    ks, vs, old = [], [], []
    for p in positions:
        kk, vv = torch.randn(s_max, G, dim, generator=g).to(DT[dt]), torch.randn(s_max, G, dim, generator=g).to(DT[dt])
        kc, vt = _pad(kk, D).transpose(0, 1).contiguous(), _pad(vv, D).permute(1, 2, 0).contiguous()
        kc[:, p:], vt[:, :, p:] = float("nan"), float("inf")
        if window and p >= window:
            vt[:, :, :p - window + 1] = float("nan")
        ks.append(kc.to(cuda)); vs.append(vt.to(cuda)); old.append((kk[:p].double(), vv[:p].double()))
    words = [torch.tensor([p], dtype=torch.int32, device=cuda) for p in positions]
    args = (tab, H, G, dim, rot, scale, eps, nw.to(cuda), nw.to(cuda), window, True, -1, n_split)
    k1, v1 = [c.clone() for c in ks], [c.clone() for c in vs]
    got = ops.decode_win(row.to(cuda), ks, vs, words, *args, waves=waves).reshape(n, H, D)
    rd = lambda x: x.to(DT[dt]).double()
    for i, p in enumerate(positions):
        qi, ki = (rd(O.rotate(O.rms_norm(x[i:i + 1], nw[:dim].double(), eps), torch.tensor([p]), r)) for x in (q, k))
        want = _attn_oracle(qi, torch.cat([old[i][0], ki]), torch.cat([old[i][1], v[i:i + 1]]), p, window, True, None, scale)
        assert _err(got[i:i + 1, :, :dim], want) < TOL[dt], p
        alone = ops.decode_win(row[i:i + 1].to(cuda), k1[i:i + 1], v1[i:i + 1], words[i:i + 1], *args).reshape(H, D)
        assert _err(got[i], alone.double().cpu()) < TOL[dt] and torch.equal(ks[i][:, p], k1[i][:, p]) and torch.equal(vs[i][:, :, p], v1[i][:, :, p])


def test_other_widths_are_refused(cuda):
    from llava_mi355x import _C, ops
    k, v = torch.zeros(2, 1, 128, 64, dtype=torch.bfloat16, device=cuda), torch.zeros(2, 1, 64, 128, dtype=torch.bfloat16, device=cuda)
    words = [torch.zeros(1, dtype=torch.int32, device=cuda) for _ in range(2)]
    with pytest.raises(_C.LmxError):
        ops.decode_win(torch.zeros(2, 3 * 64, dtype=torch.bfloat16, device=cuda), list(k), list(v), words, None, 1, 1, 64, 0, 1.0, 1e-5, sink=False, waves=6)
