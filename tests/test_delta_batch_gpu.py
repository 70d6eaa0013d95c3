"""Delta rule decode steps of batches on both sides of the line between one workgroup of 1024 threads a head (heads x sequences up to 256, where a parallel layer's mixture also chooses
its experts in the same launch) and two workgroups of 512 threads a CU past it (csrc/delta.hip): every padded head width, as many channels as threads and more, more taps than are read
at once, low-rank inputs of one, two and three pieces."""
import pytest
import torch

from oracle import vizosun_oracle as O
from test_vizosun_gpu import DT, TOL, _batch_logits
from vizosun_util import build_config, config, delta, dense, moe, rel, steady_routing

pytestmark = pytest.mark.gpu
SHAPES = {64: ([delta(8, 4, 60, 50, 4, moe(40, 5, 2)), delta(8, 8, 64, 64, 3, dense(40))], (20, 70)),
          128: ([delta(8, 2, 100, 250, 4, moe(48, 6, 3)), delta(8, 8, 128, 128, 1, None)], (140, 64)),
          256: ([delta(8, 8, 200, 70, 5, moe(24, 4, 1)), delta(8, 4, 256, 250, 4, None)], (65, 130))}
_w, _m, _o = {}, {}, {}


def weights(dk, steady):
    if (dk, steady) not in _w:
        layers, ranks = SHAPES[dk]
        cfg = config(layers, 100, 97)
        w = O.make_weights(cfg, dk, ranks)
        _w[dk, steady] = cfg, steady_routing(cfg, w) if steady else w
    return _w[dk, steady]


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("dk", list(SHAPES))
@pytest.mark.parametrize("n", [32, 33])
def test_both_forms(cuda, n, dk, dt):
    """256 and 264 heads of a layer, prompts of 1 .. 7 tokens (shorter and longer than the convolutions reach) and three steps behind each."""
    cfg, w = weights(dk, dt != "f32")
    if (dk, dt) not in _m:
        _m[dk, dt] = build_config(cfg, w, DT[dt], 64)
    ts = [torch.randint(0, 97, (4 + i % 7,), generator=torch.Generator().manual_seed(900 + i)).tolist() for i in range(n)]
    got = _batch_logits(_m[dk, dt], [t[:-3] for t in ts], [t[-3:] for t in ts])
    for i, (t, g) in enumerate(zip(ts, got)):
        if (dk, dt != "f32", i) not in _o:
            _o[dk, dt != "f32", i] = O.logits(cfg, w, t)
        assert rel(g, _o[dk, dt != "f32", i]) < TOL[dt], i
