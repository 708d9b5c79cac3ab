"""The one-pass step at sizes past the caches, where a wave's weights and momentum are loaded and stored in whole lines: each
width that has such a kernel, rows at its edges, a label count that ends inside a tile.  Against float64; the bounds are half an
fp16 step of the result (2^-11 of it) beside what G's own rounding (2^-12 of each of the batch's terms) and fp32 sums bring."""
import pytest
import torch

from renee_amd import XFCLayer, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,d", [(1, 80011, 768), (17, 76849, 768), (32, 77005, 768), (32, 60003, 1024), (9, 60031, 1024),
                                   (64, 115019, 512), (33, 117440, 512)])
def test_step_in_whole_lines(dev, B, L, d):
    lr, mu, wd, scale = 0.1, 0.9, 0.01, 2.0
    assert L * d * 4 > 224 << 20
    X = synth.make_X(B, d, 3, dev).half()
    W = (synth.make_W(L, d, 3, dev) * 20).half()
    M = (synth.make_W(L, d, 4, dev) * 0.1).half()
    P = synth.make_positives(B, L, 8, 2.3, 1.1, 3)
    px, py = (t.to(dev) for t in P.coo())
    lay = XFCLayer(L, d, B, dev, lr=lr, momentum=mu, weight_decay=wd, weight=W.clone())
    lay.momentum_buffer.copy_(M)
    print(f"step: B={B} L={L} d={d}", flush=True)
    dX = lay.xfc_backward(X, px, py, scale=scale)
    x, w, m = X.double(), W.double(), M.double()
    g = torch.sigmoid(x @ w.t())
    g[px, py] -= 1.0
    assert float((lay.outsoft[:B, :L].double() - g).abs().max()) <= 2.0 ** -12 + 1e-5
    want = scale * (g @ w)
    slack = scale * (2.0 ** -12 + 1e-5) * w.abs().sum(0)
    assert bool(((dX.double() - want).abs() <= slack).all())
    dw = g.t() @ x
    mm = mu * m + dw + wd * w
    ww = w - lr * mm
    slack = (2.0 ** -12 + 1e-5) * x.abs().sum(0) + 2.0 ** -20
    assert bool(((lay.momentum_buffer.double() - mm).abs() <= slack + 2.0 ** -11 * mm.abs()).all())
    assert bool(((lay.xfc_weight.double() - ww).abs() <= lr * slack + 2.0 ** -11 * ww.abs() + 2.0 ** -20).all())
