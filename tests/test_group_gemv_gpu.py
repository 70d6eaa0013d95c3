"""Mixtures whose rows are several pieces of 512 columns (csrc/moe.hip, group_gemv_kernel): one to six of them, taken one, two, three and four at a time, with and without columns behind
the last whole piece; decoded rows (few slots) and, in fp32, prompts (thousands of workgroups)."""
import pytest
import torch

from oracle import vizosun_oracle as O
from test_vizosun_gpu import DT, TOL, run
from vizosun_util import build_config, config, delta, moe, rel, steady_routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("width,ff", [(400, 700), (1100, 1500), (2000, 2500), (1600, 3000)])
def test_rows_of_several_pieces(cuda, width, ff, dt):
    """Gate and up rows of about `width` columns, down rows of about `ff` (padded): 1 and 2 pieces, 3 and 3, 4 and 5, 4 and 6."""
    cfg = config([delta(1, 1, 40, 48, 2, moe(ff, 5, 2))], width, 67, None, bigram=None)
    w = O.make_weights(cfg, width)
    if dt != "f32":
        w = steady_routing(cfg, w)
    m = build_config(cfg, w, DT[dt], 256)
    t = torch.randint(0, 67, (130,), generator=torch.Generator().manual_seed(ff)).tolist()
    want = O.logits(cfg, w, t)
    for cuts in ((), (120,) + tuple(range(121, 130))):
        assert rel(run(m, t, cuts), want) < TOL[dt], cuts
