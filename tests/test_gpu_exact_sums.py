"""The products' edges with whole-number operands: every product and partial sum stays below 2^24, so fp32 sums are
exact in any order and results must be equal, not close."""
import pytest
import torch

from renee_amd import XFCLayer, xfc_gemm

pytestmark = pytest.mark.gpu


def _whole(rows, cols, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(-2, 3, (rows, cols), generator=g).half()


# 32 pieces of 4 columns per workgroup of the reduction, 32 threads to a piece below 1024 workgroups and 8 from there on;
# one piece, a partial workgroup, both sides of the line; slices past the end of the contraction; row tiles of 64, 128, 256
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (3, 40, 4104), (64, 768, 20008), (100, 136, 72), (131, 992, 3000),
                                   (131, 1008, 3000), (520, 264, 70008)])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (2.0, -1.0)])
def test_split_product_and_its_reduction(dev, M, N, K, alpha, beta):
    G, W = _whole(M, K, 1), _whole(K, N, 2)
    wide = torch.full((M, N + 4), 3.0, device=dev)
    print(f"G.W: M={M} N={N} K={K} alpha={alpha} beta={beta}", flush=True)
    xfc_gemm(G.to(dev), W.to(dev), wide[:, :N], alpha, beta, False)
    want = alpha * (G.float() @ W.float()) + beta * 3.0
    assert torch.equal(wide[:, :N].cpu(), want)
    assert bool((wide[:, N:] == 3.0).all())


# logits are at most 4 * 200 and whole, so fp16 holds them; contraction lengths with a remainder, ragged rows and labels
@pytest.mark.parametrize("B,L,d", [(1, 9, 8), (65, 300, 72), (129, 257, 200), (300, 1031, 136), (513, 511, 64)])
def test_logits_at_the_edges_of_tiles(dev, B, L, d):
    X, W = _whole(B, d, 3), _whole(L, d, 4)
    layer = XFCLayer(L, d, B, dev, weight=W)
    print(f"X.W^T: B={B} L={L} d={d}", flush=True)
    assert torch.equal(layer.xfc_forward(X.to(dev)).float().cpu(), X.float() @ W.float().t())
