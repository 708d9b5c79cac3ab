"""G of a small batch and its positives in one launch: every width that has a kernel, row counts at the edges of its two sizes,
label counts around a tile of 32, both forms of the label list with repeated and dropped pairs.  Bound: half an fp16 step below
one (2^-12), and 1e-5 for the logit's fp32 sum and the exponential."""
import pytest
import torch

from renee_amd import XFCLayer, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,d", [(1, 128), (17, 256), (32, 384), (33, 384), (64, 512), (33, 768), (64, 768), (16, 768), (32, 1024),
                                 (64, 128), (50, 256)])
@pytest.mark.parametrize("L", [8, 31, 33, 4099])
def test_grad_of_a_small_batch(dev, B, d, L):
    X = synth.make_X(B, d, 1).half()
    W = (synth.make_W(L, d, 1) * 40).half()
    g = torch.Generator().manual_seed(B + L)
    n = min(2 * B, 100)
    px, py = torch.randint(0, B, (n,), generator=g), torch.randint(0, L, (n,), generator=g)
    px, py = torch.cat([px, px[:3], torch.tensor([B, 0, -1])]), torch.cat([py, py[:3], torch.tensor([0, L, 0])])
    ok = (px >= 0) & (px < B) & (py >= 0) & (py < L)
    ref = torch.sigmoid(X.double() @ W.double().t())
    hit = torch.zeros(B, L, dtype=torch.bool)
    hit[px[ok], py[ok]] = True
    want = (ref - hit.double()).to(dev)
    lay = XFCLayer(L, d, B, dev, weight=W)
    lay.outsoft.fill_(float("nan"))
    print(f"G: B={B} L={L} d={d}", flush=True)
    G = lay.fwd_grad(X.to(dev), px.to(dev), py.to(dev))
    assert float((G.double() - want).abs().max()) <= 2.0 ** -12 + 1e-5
    assert int((G < 0).sum()) == int(hit.sum())
    pad = lay.outsoft[:B, L:(L + 7) // 8 * 8]
    assert bool((pad == 0).all())
    rows = [sorted(set(py[ok & (px == b)].tolist())) for b in range(B)]
    rowptr = torch.tensor([0] + [len(r) for r in rows]).cumsum(0).to(torch.int32)
    colidx = torch.tensor([c for r in rows for c in r], dtype=torch.int32)
    lay.outsoft.fill_(float("nan"))
    assert torch.equal(lay.fwd_grad(X.to(dev), rowptr=rowptr.to(dev), colidx=colidx.to(dev)), G)


def test_many_labels_of_128_dims_go_through_the_product(dev):
    """64 rows x 131,072 x 128: one launch is the slower there.  The pass with the loss always runs the product, so that its G has
    the same bits (the other sums the logit in another order)."""
    B, L, d = 64, 131072, 128
    X, W = synth.make_X(B, d, 1, dev, torch.float32).half(), (synth.make_W(L, d, 1, dev, torch.float32) * 40).half()
    lay = XFCLayer(L, d, B, dev, weight=W)
    px, py = torch.arange(B, device=dev), torch.arange(B, device=dev) * 7
    G = lay.fwd_grad(X, px, py).clone()
    H = lay.fwd_grad(X, px, py, loss_out=torch.zeros(1, device=dev)).clone()
    assert float((G - H).abs().max()) <= 2.0 ** -11 + 2e-5
    G[px, py] = 0  # the positives' logits are summed in an order of their own
    H[px, py] = 0
    assert torch.equal(G, H)
