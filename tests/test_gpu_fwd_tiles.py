"""The forward pass by its four tiles, whichever the sizes lead to, and by large tiles with the labels that whole rounds leave by
small ones: rows and labels at the edges of 64, 128 and 256, leading dimensions past the width, against float64.  Bounds: fp32
sums of d products of halves, 2^-23 of the sum of their magnitudes per addition with a factor of four for the order, through a sigmoid
of slope 1/4 at most (and its own few fp32 roundings), and one rounding to fp16 (2^-11)."""
import pytest
import torch

from renee_amd import xfc_gemm
from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu
SUM = 4 * 2.0 ** -23
# label counts: parts of a tile, one tile of 128 and more, whole rounds of 256-label tiles and a few labels (256 CUs, 128 to 512 rows)
SIZES = [(65, 1, 72), (127, 129, 64), (128, 300, 776), (129, 127, 128), (256, 1025, 64), (257, 385, 200), (300, 8001, 768),
         (1000, 140, 64), (70, 66001, 64), (200, 65537, 128), (512, 32769, 128), (513, 22003, 64)]


def _st():
    return torch.cuda.current_stream().cuda_stream


def _inputs(dev, B, L, d, pad=8):
    g = torch.Generator(device=dev).manual_seed(B + 3 * L + 7 * d)
    X = torch.full((B, d + pad), float("nan"), device=dev, dtype=torch.float16)
    W = torch.full((L, d + pad), float("nan"), device=dev, dtype=torch.float16)
    X[:, :d] = (torch.randn(B, d, generator=g, device=dev) * 0.3).half()
    W[:, :d] = (torch.randn(L, d, generator=g, device=dev) * 0.3).half()
    x, w = X[:, :d].double(), W[:, :d].double()
    return X, W, x @ w.t().contiguous(), x.abs() @ w.abs().t().contiguous()


def _rounded(got, want, slack):
    return bool(((got.double() - want).abs() <= slack + 2.0 ** -11 * want.abs() + 2.0 ** -25).all())


@pytest.mark.parametrize("B,L,d", SIZES)
def test_logits_gradient_and_loss(dev, B, L, d):
    X, W, z, az = _inputs(dev, B, L, d)
    ldg = (L + 7) // 8 * 8 + 8
    print(f"forward: B={B} L={L} d={d}", flush=True)
    out = torch.full((B, ldg), 7.0, device=dev, dtype=torch.float16)
    check(lib().xfc_logits(X.data_ptr(), d + 8, W.data_ptr(), d + 8, out.data_ptr(), ldg, B, L, d, _st()), "xfc_logits")
    assert _rounded(out[:, :L], z, SUM * az) and bool((out[:, L:] == 7.0).all())

    pairs = torch.tensor([[0, 0], [B - 1, L - 1], [B // 2, L // 2], [B - 1, 0], [B // 2, L // 2]], device=dev)  # one of them twice
    px, py = pairs[:, 0].contiguous(), pairs[:, 1].contiguous()
    y = torch.zeros(B, L, device=dev, dtype=torch.float64)
    y[px, py] = 1.0
    want = torch.sigmoid(z) - y
    terms = torch.nn.functional.softplus(z) - y * z
    ws = torch.empty(lib().xfc_fwd_grad_workspace_bytes(L, 5), dtype=torch.uint8, device=dev)
    for loss in (None, torch.full((1,), float("nan"), device=dev)):
        G = torch.full((B, ldg), 7.0, device=dev, dtype=torch.float16)
        check(lib().xfc_fwd_grad_coo(X.data_ptr(), d + 8, W.data_ptr(), d + 8, px.data_ptr(), py.data_ptr(), 5, G.data_ptr(), ldg, B, L, d,
                                     None if loss is None else loss.data_ptr(), ws.data_ptr(), ws.numel(), _st()), "xfc_fwd_grad_coo")
        assert _rounded(G[:, :L], want, 0.25 * SUM * az + 2.0 ** -21)
        assert bool((G[:, L:ldg - 8] == 0.0).all()) and bool((G[:, ldg - 8:] == 7.0).all())
        if loss is not None:  # terms summed in double: each off by its sum's error and a few roundings of 1 + e^-|z| and its logarithm
            slack = float((SUM * az + 2.0 ** -21).sum())
            assert abs(float(loss) - float(terms.sum())) <= slack + 2.0 ** -23 * float(terms.sum())


@pytest.mark.parametrize("B,L,d", [(128, 304, 776), (256, 1032, 64), (512, 32776, 128)])
def test_alpha_and_beta(dev, B, L, d):
    X, W, z, az = _inputs(dev, B, L, d, 0)
    for beta in (0.0, 0.5):
        out = torch.rand(B, L, device=dev).half()
        want = torch.sigmoid(0.5 * z + beta * out.double())
        print(f"sigmoid: B={B} L={L} d={d} beta={beta}", flush=True)
        xfc_gemm(X, W.t(), out, 0.5, beta, True)
        assert _rounded(out, want, 0.25 * (0.5 * SUM * az + 2.0 ** -22) + 2.0 ** -21)


# enough labels for the maxima of blocks of 32: small tiles, large ones, and both
@pytest.mark.parametrize("B,L,d", [(100, 90001, 64), (256, 131072, 64), (512, 98305, 128), (300, 70003, 72)])
def test_best_of_the_logits(dev, B, L, d):
    X, W, _, _ = _inputs(dev, B, L, d, 0)
    K = 20
    z = torch.empty(B, (L + 7) // 8 * 8, device=dev, dtype=torch.float16)
    check(lib().xfc_logits(X.data_ptr(), d, W.data_ptr(), d, z.data_ptr(), z.stride(0), B, L, d, _st()), "xfc_logits")
    logits = torch.empty(lib().xfc_topk_workspace_bytes(B, L, K), dtype=torch.uint8, device=dev)
    maxima = torch.full((B * ((L + 255) // 256 * 8) * 2,), 255, dtype=torch.uint8, device=dev)
    v, i = torch.empty(B, K, device=dev), torch.empty(B, K, device=dev, dtype=torch.int64)
    print(f"top-{K}: B={B} L={L} d={d}", flush=True)
    check(lib().xfc_topk_scratch(X.data_ptr(), d, W.data_ptr(), d, B, L, d, L, K, v.data_ptr(), i.data_ptr(), logits.data_ptr(), logits.numel(),
                                 maxima.data_ptr(), maxima.numel(), _st()), "xfc_topk_scratch")
    want = torch.sort(z[:, :L].float(), dim=1, descending=True, stable=True)
    assert torch.equal(v, want.values[:, :K]) and torch.equal(i, want.indices[:, :K])
