"""The pass that applies the label list to G after the product, and what it contributes to the loss: pairs listed more
than once, neighbours that share a 32-bit word of G, pairs out of range, long lists, and the row search of a CSR list.
Against float64."""
import pytest
import torch

from renee_amd import XFCLayer, synth

pytestmark = pytest.mark.gpu


def _check(dev, X, W, Y, coo=None, csr=None):
    """G within its rounding to fp16 (|G| <= 1), below zero exactly at the pairs; the loss within the rounding of its
    groups of terms and of itself to fp32 (a pair counted twice or not at all is 1e-5 of it and more)."""
    (B, d), L = X.shape, W.shape[0]
    n = coo[0].numel() if coo else csr[1].numel()
    lay = XFCLayer(L, d, B, dev, weight=W, max_positives=max(n, 1))
    print(f"positives: B={B} L={L} nnz={n} csr={csr is not None}", flush=True)
    kw = dict(pos_x=coo[0].to(dev), pos_y=coo[1].to(dev)) if coo else dict(rowptr=csr[0].to(dev), colidx=csr[1].to(dev))
    Z = X.double() @ W.double().t()
    want = torch.sigmoid(Z) - Y.double()
    bce = float(torch.nn.functional.binary_cross_entropy_with_logits(Z, Y.double(), reduction="sum"))
    loss = torch.zeros(1, device=dev)
    for loss_out in (None, loss):
        lay.outsoft.fill_(9.0)
        G = lay.fwd_grad(X.to(dev), loss_out=loss_out, **kw).cpu()
        assert torch.equal(torch.signbit(G), Y)
        assert (G.double() - want).abs().max() <= 2.0 ** -11 + 1e-5
    assert abs(float(loss) - bce) <= 2.0 ** -21 * bce


# the three row tiles, whose logits are summed in two different orders
@pytest.mark.parametrize("B", [40, 100, 300])
@pytest.mark.parametrize("csr", [False, True])
def test_repeated_neighbouring_and_dropped_pairs(dev, B, csr):
    L, d = 203, 128
    g = torch.Generator().manual_seed(B)
    X, W = synth.make_X(B, d, B).half(), (synth.make_W(L, d, B) * 20).half()
    rows, cols = [], []
    for r in range(0, B, 3):
        c = int(torch.randint(0, L - 4, (1,), generator=g))
        mine = [c, c + 1, c + 2, c + 3] * 3 + [c] * 5 + [0, L - 1]     # both halves of a word, two neighbouring words
        mine += [-1, L, 2 ** 31 - 1] if r % 2 else []
        mine = [mine[int(i)] for i in torch.randperm(len(mine), generator=g)]
        rows += [r] * len(mine)
        cols += mine
    px, py = torch.tensor(rows), torch.tensor(cols)
    Y = torch.zeros(B, L, dtype=torch.bool)
    keep = (py >= 0) & (py < L)
    Y[px[keep], py[keep]] = True
    if csr:
        ptr = torch.zeros(B + 1, dtype=torch.int32)
        ptr[1:] = torch.bincount(px, minlength=B).cumsum(0).int()
        _check(dev, X, W, Y, csr=(ptr, py.int()))
    else:
        mix = torch.randperm(len(rows) + 3, generator=g)   # any order, and rows out of range
        px = torch.cat([px, torch.tensor([-1, B, 2 ** 40])])[mix]
        py = torch.cat([py, torch.tensor([0, 0, 0])])[mix]
        _check(dev, X, W, Y, coo=(px, py))


@pytest.mark.parametrize("csr", [False, True])
def test_more_pairs_than_waves(dev, csr):
    """70,000 pairs, a good part of them repeated; the pass launches 65,536 waves at most."""
    B, L, d, per = 700, 300, 64, 100
    X, W = synth.make_X(B, d, 5).half(), (synth.make_W(L, d, 5) * 20).half()
    py = torch.randint(0, L, (B, per), generator=torch.Generator().manual_seed(5))
    Y = torch.zeros(B, L, dtype=torch.bool).scatter_(1, py, True)
    if csr:
        _check(dev, X, W, Y, csr=(torch.arange(0, B * per + 1, per, dtype=torch.int32), py.flatten().int()))
    else:
        _check(dev, X, W, Y, coo=(torch.arange(B).repeat_interleave(per), py.flatten()))


# the search takes 64 row pointers at a time: one round up to 64 rows, two up to 4096, three above
@pytest.mark.parametrize("B", [1, 2, 63, 64, 65, 129, 4095, 4096, 4097, 4200])
def test_row_search(dev, B):
    L, d = 41, 32
    g = torch.Generator().manual_seed(B)
    X, W = synth.make_X(B, d, B).half(), (synth.make_W(L, d, 1) * 20).half()
    for fill in (1.0, 0.3, 0.01):   # rows with labels; the rest are empty, at both ends and in long runs
        Y = (torch.rand(B, L, generator=g) < 0.1) & (torch.rand(B, 1, generator=g) < fill)
        if fill < 1.0 and B > 2:
            Y[0] = Y[-1] = False
        Y[B // 2, 3] = True
        ptr = torch.zeros(B + 1, dtype=torch.int32)
        ptr[1:] = Y.sum(1).cumsum(0).int()
        _check(dev, X, W, Y, csr=(ptr, Y.nonzero()[:, 1].int()))
