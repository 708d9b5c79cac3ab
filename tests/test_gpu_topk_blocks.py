"""The K <= 8 scorer's two kernels at the sizes where they can go wrong: units and blocks past the label count, widths that
do not fill a k-step or a piece of steps, rows past the batch, more blocks than the second kernel keeps in registers, label
ranges when the workspace is short, and scores that are no numbers.  Operands are small whole numbers, so that every score is
exact in fp32 whatever the order of its sum, and values and labels have to be those of a stable sort."""
import pytest
import torch

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _run(X, W, K, numy=None, ws_bytes=None):
    h = lib()
    B, d = X.shape
    L = W.shape[0]
    nbytes = h.xfc_topk_workspace_bytes(B, L, K) if ws_bytes is None else ws_bytes
    ws = torch.empty(nbytes, dtype=torch.uint8, device=X.device)
    v = torch.full((B, K), float("nan"), device=X.device)
    i = torch.full((B, K), -1, dtype=torch.int64, device=X.device)
    print(f"top-{K}: B={B} L={L} d={d} workspace={nbytes}", flush=True)
    check(h.xfc_topk(X.data_ptr(), X.stride(0), W.data_ptr(), W.stride(0), B, L, d, L if numy is None else numy, K,
                     v.data_ptr(), i.data_ptr(), ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream), "xfc_topk")
    return v, i


def _expect(X, W, K):
    Z = X.float() @ W.float().t()
    # whole numbers below 2^20 and label ids below 2^23: (score, label) as one exact double
    order = (Z.double() * 2.0 ** 23 - torch.arange(W.shape[0], dtype=torch.float64, device=Z.device)).topk(K, dim=1).indices
    return Z.gather(1, order), order


def _problem(dev, B, L, d, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randint(-2, 3, (B, d), generator=g).half().to(dev), torch.randint(-2, 3, (L, d), generator=g).half().to(dev))


# widths: below a k-step, one step and a tail, a piece of four steps and a tail, and (3000) more than the LDS holds rows of
@pytest.mark.parametrize("B,L,d,K", [(1, 17, 8, 8), (16, 16, 40, 5), (17, 1000, 136, 5), (33, 4111, 264, 8), (64, 65, 1288, 3),
                                     (20, 3001, 3000, 5), (16, 3001, 3000, 5), (64, 9000, 32, 1), (65, 257, 40, 8), (128, 70001, 136, 5),
                                     (129, 513, 72, 5), (700, 12345, 64, 5),
                                     # runs of two and four units; more than 131,072 blocks
                                     (16, 131077, 64, 5), (20, 270011, 64, 5), (40, 700001, 8, 5), (3, 2200003, 8, 8), (2, 290001, 768, 5), (9, 290001, 768, 5)])
def test_blocks_against_a_stable_sort(dev, B, L, d, K):
    X, W = _problem(dev, B, L, d, B + L + d)
    v, i = _run(X, W, K)
    ev, ei = _expect(X, W, K)
    assert torch.equal(v, ev) and torch.equal(i, ei)


@pytest.mark.parametrize("B,L,d,K", [(16, 5003, 64, 5), (32, 40000, 72, 1), (96, 40000, 64, 8), (300, 9001, 64, 5)])
def test_a_short_workspace_takes_the_labels_in_ranges(dev, B, L, d, K):
    """From the least that is accepted on, the K best of a range are carried to the next; ties still go to the lower label."""
    X, W = _problem(dev, B, L, d, B + K)
    ev, ei = _expect(X, W, K)
    full, least = lib().xfc_topk_workspace_bytes(B, L, K), 8 * B * K * 8 + (B + 3) // 4 * 16
    for nbytes in (least, least + 4 * 48 * B, full - 16):
        v, i = _run(X, W, K, ws_bytes=nbytes)
        assert torch.equal(v, ev) and torch.equal(i, ei)


@pytest.mark.parametrize("B", [5, 70, 200])
def test_scores_that_are_no_numbers_are_passed_over(dev, B):
    """Blocks whose scores are all NaN, a block that holds NaN beside the best scores, -inf everywhere else: the finite ones
    first, then -inf in label order, and (-inf, numy - 1) where no label is left."""
    L, d, K = 3000, 8, 8
    nan, inf = float("nan"), float("inf")
    W = torch.zeros(L, d)
    W[:, 0] = -inf
    W[0:1500, 0] = nan
    W[100, 0], W[2047, 0], W[2999, 0] = 2.0, 3.0, 3.0
    X = torch.zeros(B, d)
    X[:, 0] = 1.0
    W[:, 1:] = 0.0
    Xd, Wd = X.half().to(dev), W.half().to(dev)
    v, i = _run(Xd, Wd, K)
    assert i.cpu().tolist() == [[2047, 2999, 100, 1500, 1501, 1502, 1503, 1504]] * B
    assert v.cpu()[:, :3].tolist() == [[3.0, 3.0, 2.0]] * B and bool(torch.isneginf(v[:, 3:]).all())
    W[1500:, 0] = nan
    W[2047, 0] = 3.0
    v, i = _run(Xd, W.half().to(dev), K, numy=2500)
    assert i.cpu().tolist() == [[2047, 100] + [2499] * 6] * B
    assert v.cpu()[:, :2].tolist() == [[3.0, 2.0]] * B and bool(torch.isneginf(v[:, 2:]).all())


@pytest.mark.parametrize("B", [1, 3])
def test_label_counts_at_the_end_of_32_bits(dev, B):
    """The largest label count there is, in ranges: the last label, one on each side of a range's end, and ties to the lower."""
    L, d, K = 2 ** 31 - 1, 8, 6
    if torch.cuda.mem_get_info()[0] < 45 << 30:
        pytest.skip("needs 45 GB")
    W = torch.zeros(L, d, dtype=torch.float16, device=dev)
    best = {L - 1: 4.0, 2 ** 30 - 1: 3.0, 2 ** 30: 3.0, 5: 2.0}
    for label, score in best.items():
        W[label, 0] = score
    X = torch.zeros(B, d, dtype=torch.float16, device=dev)
    X[:, 0] = 1.0
    v, i = _run(X, W, K)
    assert i.cpu().tolist() == [[L - 1, 2 ** 30 - 1, 2 ** 30, 5, 0, 1]] * B
    assert v.cpu().tolist() == [[4.0, 3.0, 3.0, 2.0, 0.0, 0.0]] * B


def test_a_width_whose_fragments_exceed_32_bits_of_bytes(dev):
    """2^25 dims, 17 rows: X as fragments would take 2 GB, no LDS and no positive int; the main loop takes the call."""
    B, L, d, K = 17, 3, 2 ** 25, 3
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    X, W = torch.zeros(B, d, dtype=torch.float16, device=dev), torch.zeros(L, d, dtype=torch.float16, device=dev)
    at = torch.randint(0, d, (64,), generator=g, device=dev)
    at[0] = d - 1
    X[:, at] = torch.randint(-2, 3, (B, 64), generator=g, device=dev).half()
    W[:, at] = torch.randint(-2, 3, (L, 64), generator=g, device=dev).half()
    v, i = _run(X, W, K)
    ev, ei = _expect(X[:, at.unique()], W[:, at.unique()], K)
    assert torch.equal(v, ev) and torch.equal(i, ei)


# streamed past 16 and 32 rows, the main loop on 128 and 256; widths that end inside a k-step of 32 and a stage of 64
@pytest.mark.parametrize("B,L,d", [(7, 4001, 72), (16, 20011, 768), (32, 5003, 200), (20, 9001, 1032), (40, 9001, 104), (128, 7001, 768),
                                   (129, 5003, 136), (300, 9001, 776)])
def test_the_second_look_has_the_bits_of_the_first(dev, B, L, d):
    """What the K best blocks rest on: a row's best score, formed again, is the largest of the maxima to the last bit.  Operands whose
    sums round; with K = 1 and room for all maxima these lie at the start of the workspace."""
    g = torch.Generator().manual_seed(B + d)
    X, W = torch.randn(B, d, generator=g).half().to(dev), torch.randn(L, d, generator=g).half().to(dev)
    h = lib()
    small = B <= 32 and -(-d // 32) * (1024 if B <= 16 else 2048) <= 160 * 1024
    blocks = -(-L // 16) if small else -(-L // 256) * 8
    ldb = -(-blocks // 4) * 4
    nbytes = max(h.xfc_topk_workspace_bytes(B, L, 1), B * ldb * 4)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    v, i = torch.empty(B, 1, device=dev), torch.empty(B, 1, dtype=torch.int64, device=dev)
    print(f"bits: B={B} L={L} d={d}", flush=True)
    check(h.xfc_topk(X.data_ptr(), d, W.data_ptr(), d, B, L, d, L, 1, v.data_ptr(), i.data_ptr(), ws.data_ptr(), nbytes,
                     torch.cuda.current_stream().cuda_stream), "xfc_topk")
    maxima = ws.view(torch.float32)[:B * ldb].view(B, ldb)[:, :-(-L // (16 if small else 32))]
    assert torch.equal(maxima.max(dim=1).values, v[:, 0])
    z = X.double() @ W.double().t()
    assert float((z.max(dim=1).values - v[:, 0].double()).abs().max()) <= 1e-5 * float(z.abs().max())
