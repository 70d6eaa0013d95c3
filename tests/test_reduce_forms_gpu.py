"""Column sums and the cross-entropy's forward at the edges of their forms (csrc/train.hip): row and column remainders, rows in whole 16-byte loads and not, logits of -inf;
several images' attention in one launch (csrc/attention.hip) against one launch an image.  Against float64; the bounds are those of fp32 sums of the lengths at hand."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,cols,ld,off", [(1, 8, 8, 0), (127, 64, 64, 0), (129, 72, 80, 0), (1000, 4096, 4096, 0), (300, 63, 70, 0), (515, 128, 136, 3), (16, 200, 200, 0)])
def test_col_sum(cuda, dt, rows, cols, ld, off):
    from llava_mi355x import ops
    g = torch.Generator().manual_seed(rows + cols)
    buf = torch.randn(rows * ld + off + 8, generator=g).to(dt).to(cuda)
    dy = buf[off:off + rows * ld].view(rows, ld)[:, :cols]
    want = dy.double().sum(0)
    bound = rows * 2.0 ** -24 * dy.double().abs().sum(0) + 1e-30
    out = torch.full((cols,), float("nan"), device=cuda)
    ops.check(ops.lib.lmx_op_col_sum(ops.torch_dtype_code(dt), ops.ptr(buf[off:]), ld, rows, cols, ops.ptr(out), ops.stream_handle()), "col_sum")
    assert bool(((out.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [1, 7, 8, 255, 2047, 2048, 2056, 32003])
def test_ce_rows(cuda, dt, V):
    from llava_mi355x import ops
    g = torch.Generator().manual_seed(V)
    logits = (torch.randn(2, 5, V, generator=g) * 8).to(dt)
    if V > 8:
        logits[0, 1, 1:] = float("-inf")                      # one finite logit: its lane alone has a sum
        logits[1, 2, ::3] = float("-inf")
    labels = torch.zeros(2, 5, dtype=torch.int64)
    x = logits.double()[:, :-1].reshape(-1, V)
    want = (torch.logsumexp(x, 1) - x[:, 0])
    want = want[torch.isfinite(want)].sum() if V <= 8 else want
    if V > 8:
        labels[1, 3] = -100                                   # the row whose label logit is -inf
        keep = torch.ones(8, dtype=torch.bool); keep[4 + 2] = False
        want = want[keep].mean()
    else:
        want = want / 8
    loss, _, _ = ops.ce_loss(logits.to(cuda), labels.to(cuda))
    assert abs(loss.item() - want.item()) <= 2.0 ** -23 * (V / 256 + 64 + 4 * x[torch.isfinite(x)].abs().max().item())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [2, 5])
def test_images_together_as_apart(cuda, dt, n):
    """A wrong image's rows, keys or values would be as far off as two images are from each other; the linears' forms may differ with the rows, so a few roundings are allowed."""
    from synthetic import build as harness, recipes as synth
    cfg = synth.CONFIGS["tiny"]
    model = harness.build_model(cfg, dtype=dt, seed=0)
    pix = torch.from_numpy(synth.make_pixels(cfg, n, seed=11)).to(cuda, dt)
    both = model.encode_images(pix)
    alone = torch.cat([model.encode_images(pix[i:i + 1]) for i in range(n)])
    apart = (both[0] - both[1]).abs().max().item()
    assert (both - alone).abs().max().item() <= 0.1 * apart
