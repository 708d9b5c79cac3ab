"""Top-K up to 8 with lists, the pass for workspaces that are short of the maxima: each row tile, with and without bounds from a
sample, from the least workspace on; scores that are no numbers and -inf; the same bits as the pass by maxima."""
import pytest
import torch

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _run(X, W, K, nbytes, numy=None):
    B, d = X.shape
    L = W.shape[0]
    ws = torch.empty(nbytes, dtype=torch.uint8, device=X.device)
    v = torch.full((B, K), float("nan"), device=X.device)
    i = torch.full((B, K), -1, dtype=torch.int64, device=X.device)
    print(f"top-{K}: B={B} L={L} d={d} workspace={nbytes}", flush=True)
    check(lib().xfc_topk(X.data_ptr(), d, W.data_ptr(), d, B, L, d, L if numy is None else numy, K, v.data_ptr(), i.data_ptr(),
                         ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream), "xfc_topk")
    return v, i


def _least(B, K):
    return 64 * B * K + (B + 3) // 4 * 16


def _sizes(B, L, K):
    """The least, one that adds label groups, one that also has room for the sample, all short of a third of the maxima."""
    full = lib().xfc_topk_workspace_bytes(B, L, K)
    return [n for n in (_least(B, K), 3 * _least(B, K) + 16, _least(B, K) + B * (4096 + 12 * K) + 16) if 4 * n < full]


def _expect(X, W, K):
    Z = X.float() @ W.float().t()
    order = (Z.double() * 2.0 ** 23 - torch.arange(W.shape[0], dtype=torch.float64, device=Z.device)).topk(K, dim=1).indices
    return Z.gather(1, order), order


# whole numbers: every score is exact, ties are many
@pytest.mark.parametrize("B,L,d,K", [(1, 70001, 64, 1), (64, 30000, 72, 8), (16, 300001, 24, 5), (65, 140001, 136, 5), (128, 90001, 32, 3),
                                     (129, 170001, 40, 8), (700, 133333, 64, 5)])
def test_lists_against_a_stable_sort(dev, B, L, d, K):
    g = torch.Generator().manual_seed(B + L)
    X, W = torch.randint(-2, 3, (B, d), generator=g).half().to(dev), torch.randint(-2, 3, (L, d), generator=g).half().to(dev)
    ev, ei = _expect(X, W, K)
    sizes = _sizes(B, L, K)
    assert sizes
    for nbytes in sizes:
        v, i = _run(X, W, K, nbytes)
        assert torch.equal(v, ev) and torch.equal(i, ei)


@pytest.mark.parametrize("B", [5, 70, 200])
@pytest.mark.parametrize("L", [9000, 70000])  # the longer one starts from bounds
def test_scores_that_are_no_numbers_and_minus_infinity(dev, B, L):
    """As with the maxima: what is no number is never listed, -inf is, in label order, and (-inf, numy - 1) where no label is left."""
    d, K = 8, 8
    nan, inf = float("nan"), float("inf")
    W = torch.zeros(L, d)
    W[:, 0] = -inf
    W[0:1500, 0] = nan
    W[100, 0], W[2047, 0], W[L - 1, 0] = 2.0, 3.0, 3.0
    X = torch.zeros(B, d, dtype=torch.float16, device=dev)
    X[:, 0] = 1.0
    for nbytes in _sizes(B, L, K):
        v, i = _run(X, W.half().to(dev), K, nbytes)
        assert i.cpu().tolist() == [[2047, L - 1, 100, 1500, 1501, 1502, 1503, 1504]] * B
        assert v.cpu()[:, :3].tolist() == [[3.0, 3.0, 2.0]] * B and bool(torch.isneginf(v[:, 3:]).all())
    W[1500:, 0] = nan
    W[2047, 0] = 3.0
    for nbytes in _sizes(B, L, K):
        v, i = _run(X, W.half().to(dev), K, nbytes, numy=2500)
        assert i.cpu().tolist() == [[2047, 100] + [2499] * 6] * B
        assert v.cpu()[:, :2].tolist() == [[3.0, 2.0]] * B and bool(torch.isneginf(v[:, 2:]).all())
    W = torch.rand(L, d, generator=torch.Generator().manual_seed(1))
    W[:, 1:] = 0.0
    W[3, 0], W[7, 0], W[2000, 0], W[5000, 0] = nan, inf, nan, nan  # in the sample and past it
    Wd = W.half().to(dev)
    full = lib().xfc_topk_workspace_bytes(B, L, K)
    want = _run(X, Wd, K, full)
    assert want[1][:, 0].cpu().tolist() == [7] * B
    for nbytes in _sizes(B, L, K):
        v, i = _run(X, Wd, K, nbytes)
        assert torch.equal(v, want[0]) and torch.equal(i, want[1])


@pytest.mark.parametrize("B,L,d,K", [(16, 60001, 768, 5), (64, 60001, 200, 8), (100, 90001, 136, 5), (300, 120001, 384, 5)])
def test_the_bits_are_those_of_the_maxima(dev, B, L, d, K):
    g = torch.Generator().manual_seed(B)
    X, W = torch.randn(B, d, generator=g).half().to(dev), torch.randn(L, d, generator=g).half().to(dev)
    v, i = _run(X, W, K, lib().xfc_topk_workspace_bytes(B, L, K))
    for nbytes in _sizes(B, L, K):
        w, j = _run(X, W, K, nbytes)
        assert torch.equal(v, w) and torch.equal(i, j)


@pytest.mark.parametrize("B", [1, 33, 100])
def test_the_best_of_very_many_labels(dev, B):
    """K = 1 goes by lists there whatever the workspace, K = 4 by maxima."""
    L, d = 1250007, 256
    g = torch.Generator(device=dev)
    g.manual_seed(B)
    X, W = torch.randn(B, d, generator=g, device=dev).half(), torch.randn(L, d, generator=g, device=dev).half()
    v, i = _run(X, W, 1, lib().xfc_topk_workspace_bytes(B, L, 1))
    w, j = _run(X, W, 4, lib().xfc_topk_workspace_bytes(B, L, 4))
    assert torch.equal(v, w[:, :1]) and torch.equal(i, j[:, :1])


# a workspace for all label groups (256 CUs) and the sample; K = 1 goes by lists at the last size whatever it is
@pytest.mark.parametrize("B,L,K,groups", [(40, 540001, 1, 256), (100, 540001, 1, 256), (128, 540001, 3, 256), (129, 540001, 1, 256),
                                          (700, 170001, 3, 80), (100, 1250007, 1, 0)])
def test_bounds_from_a_sample_where_products_cancel(dev, B, L, K, groups):
    """Scores of identical labels, each the sum of products and of their negatives: none is more than what the sums round off, so that
    a sample summed in another order than the lists might lie above every one of them.  The first labels win, whatever they score."""
    d = 256
    g = torch.Generator().manual_seed(B)
    x, w, order = torch.randn(B, d // 2, generator=g).half() * 8, torch.randn(d // 2, generator=g).half() * 8, torch.randperm(d // 2, generator=g)
    X = torch.cat([x, -x[:, order]], 1).to(dev)
    W = torch.cat([w, w[order]]).to(dev).repeat(L, 1)
    magnitude = X.double().abs() @ W[0].double().abs()
    assert float((X.double() @ W[0].double()).abs().max()) < 1e-9  # of the order of its own roundings
    full = lib().xfc_topk_workspace_bytes(B, L, K)
    nbytes = groups * B * K * 8 + (B + 3) // 4 * 16 + B * (4096 + 12 * K) + 16 if groups else full
    assert not groups or (-(-L // 256) >= 8 * groups and 3 * nbytes < full)
    v, i = _run(X, W, K, nbytes)
    assert torch.equal(i, torch.arange(K, device=dev).expand(B, K))
    assert bool((v.double().abs() <= 4 * 2.0 ** -23 * magnitude[:, None]).all()) and float(v.abs().max()) > 0


def test_the_least_workspace_costs_label_groups_and_not_launches(dev):
    """16 rows x 700,001 x 768, K = 1 in 1,088 bytes: 18 times what it takes with 2.8 MB.  (Range after range of labels: 300 times.)"""
    B, L, d, K = 16, 700001, 768, 1
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    X, W = torch.randn(B, d, generator=g, device=dev).half(), torch.randn(L, d, generator=g, device=dev).half()
    took = []
    for nbytes in (lib().xfc_topk_workspace_bytes(B, L, K), _least(B, K)):
        _run(X, W, K, nbytes)
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(3):
            _run(X, W, K, nbytes)
        end.record()
        torch.cuda.synchronize()
        took.append(start.elapsed_time(end))
    assert took[1] < 60 * took[0]
