"""The K > 8 selection by the maxima of blocks of 32 logits, on each row tile of the forward pass: the same answer as a stable
sort of the logits, with and without the second buffer, where the maxima give a loose bound and where they give none."""
import pytest
import torch

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _run(X, W, K, scratch):
    h = lib()
    B, d = X.shape
    L = W.shape[0]
    nbytes = h.xfc_topk_workspace_bytes(B, L, K)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=X.device)
    sc = torch.empty(B * ((L + 255) // 256) * 16, dtype=torch.uint8, device=X.device)
    v = torch.empty(B, K, device=X.device)
    i = torch.empty(B, K, dtype=torch.int64, device=X.device)
    print(f"top-{K}: B={B} L={L} d={d} scratch={scratch}", flush=True)
    check(h.xfc_topk_scratch(X.data_ptr(), d, W.data_ptr(), d, B, L, d, L, K, v.data_ptr(), i.data_ptr(), ws.data_ptr(), nbytes,
                             sc.data_ptr() if scratch else None, sc.numel() if scratch else 0,
                             torch.cuda.current_stream().cuda_stream), "xfc_topk_scratch")
    return v, i


def _key(z):
    """fp16 logits as integers in the order of the selection: by value, what is no number by its bit pattern."""
    b = z.view(torch.int16).to(torch.int32) & 0xffff
    b = torch.where(b == 0x8000, torch.zeros_like(b), b)
    return torch.where(b >= 0x8000, 0xffff - b, b + 0x8000)


def _check(X, W, K):
    B, d = X.shape
    L = W.shape[0]
    Z = torch.empty(B, (L + 7) // 8 * 8, dtype=torch.float16, device=X.device)
    check(lib().xfc_logits(X.data_ptr(), d, W.data_ptr(), d, Z.data_ptr(), Z.shape[1], B, L, d,
                           torch.cuda.current_stream().cuda_stream), "xfc_logits")
    Z = Z[:, :L].contiguous()
    order = (_key(Z).double() * 2.0 ** 24 - torch.arange(L, dtype=torch.float64, device=Z.device)).topk(K, dim=1).indices
    want = Z.gather(1, order).float()
    for scratch in (True, False):
        v, i = _run(X, W, K, scratch)
        assert torch.equal(i, order)
        assert torch.equal(v.nan_to_num(nan=7e4), want.nan_to_num(nan=7e4))


# rows of each tile and past it; label counts that end inside a block, a piece of eight and a tile; K at half the blocks
@pytest.mark.parametrize("B,L,d,K", [(1, 65505, 8, 10), (64, 65543, 64, 100), (65, 70003, 40, 100), (128, 70001, 64, 9),
                                     (129, 65536 + 33, 72, 100), (300, 65537, 64, 200), (5, 70001, 64, 1000), (3, 150007, 32, 2000)])
def test_blocks_of_logits_against_a_stable_sort(dev, B, L, d, K):
    g = torch.Generator().manual_seed(B + L)
    _check(torch.randn(B, d, generator=g).half().to(dev), torch.randn(L, d, generator=g).half().to(dev), K)


@pytest.mark.parametrize("B", [3, 100, 200])
def test_loose_bounds_and_rows_without_one(dev, B):
    """Scores as given: many in few blocks (the bound leaves more than can be sorted), all equal, NaN of either sign, -inf."""
    L, K = 70009, 100
    g = torch.Generator().manual_seed(5)
    X = torch.zeros(B, 8)
    X[:, 0] = 1.0
    scores = []
    s = torch.rand(L, generator=g)
    s[1600:1600 + 32 * 99] = 2.0 + torch.rand(32 * 99, generator=g)  # 99 blocks hold 3,168 large ones: the bound is below 1
    scores.append(s)
    scores.append(torch.full((L,), 0.5))
    s = torch.rand(L, generator=g) - 0.5
    s[777], s[31000] = float("nan"), float("inf")
    scores.append(s)
    s = torch.full((L,), -float("inf"))
    s[::1001] = 1.0
    scores.append(s)
    for s in scores:
        W = torch.zeros(L, 8)
        W[:, 0] = s
        _check(X.half().to(dev), W.half().to(dev), K)
    W = torch.zeros(L, 8)
    W[:, 0] = torch.rand(L, generator=g)
    W16 = W.half()
    W16.view(torch.int16)[5000:5040, 0] = -512 + 5  # 0xfe05: no number, sign set
    _check(X.half().to(dev), W16.to(dev), K)


# more blocks at the bound than the small list holds, at its most, and more than the maxima are used for; NaN on top
@pytest.mark.parametrize("B,L,K", [(3, 300007, 2049), (2, 400009, 4096), (2, 400009, 6144), (1, 600011, 6145), (1, 700001, 8192)])
def test_long_lists_of_blocks(dev, B, L, K):
    g = torch.Generator().manual_seed(K)
    X, W = torch.randn(B, 16, generator=g).half().to(dev), torch.randn(L, 16, generator=g).half().to(dev)
    _check(X, W, K)
    W[777] = float("nan")
    _check(X, W, K)
    W[:, 1:] = 0.0  # many ties
    W[:, 0] = torch.randint(-40, 40, (L,), generator=g).half().to(dev)
    _check(X, W, K)


@pytest.mark.parametrize("K,used", [(1024, True), (6144, True), (6145, False), (8192, False)])
def test_maxima_are_made_where_they_serve(dev, K, used):
    """A selection whose list of blocks could not hold K does not pay for the maxima: the second buffer stays as it was."""
    B, L, d = 2, 600011, 16
    g = torch.Generator().manual_seed(1)
    X, W = torch.randn(B, d, generator=g).half().to(dev), torch.randn(L, d, generator=g).half().to(dev)
    h = lib()
    ws = torch.empty(h.xfc_topk_workspace_bytes(B, L, K), dtype=torch.uint8, device=dev)
    sc = torch.full((B * ((L + 255) // 256) * 16,), 0x5a, dtype=torch.uint8, device=dev)
    v, i = torch.empty(B, K, device=dev), torch.empty(B, K, dtype=torch.int64, device=dev)
    check(h.xfc_topk_scratch(X.data_ptr(), d, W.data_ptr(), d, B, L, d, L, K, v.data_ptr(), i.data_ptr(), ws.data_ptr(), ws.numel(),
                             sc.data_ptr(), sc.numel(), torch.cuda.current_stream().cuda_stream), "xfc_topk_scratch")
    assert bool((sc != 0x5a).any()) == used
