"""The gradient by itself and the updates where what is written is more than the caches hold and is stored past them, against float64:
label counts and widths that are no whole tiles, leading dimensions past the width, a gradient that is added to.  Bounds as in
test_gpu_back_step.py: fp32 sums of up to B products of halves, relative to the sums of their magnitudes, 2^-23 per addition with a
factor of four for the order; a few fp32 roundings of the update on top (2^-22), and one to fp16 (2^-11) where the result is."""
import pytest
import torch
from test_gpu_back_step import SUM, _st

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu
LR, MU, WD = 0.1, 0.9, 0.01
CHUNK = 1 << 15


def _normal(dev, seed, rows, ld, d, scale, dtype):
    """rows x ld, the columns past d filled with what no result may touch."""
    g = torch.Generator(device=dev).manual_seed(seed)
    t = torch.full((rows, ld), 7.0, device=dev, dtype=dtype)
    t[:, :d] = (torch.randn(rows, d, generator=g, device=dev) * scale).to(dtype)
    return t


def _gradient(G, X, d, l0, l1):
    g, x = G[:, l0:l1].double(), X[:, :d].double()
    return g.t().contiguous() @ x, g.abs().t().contiguous() @ x.abs()


def _inputs(dev, B, L, d):
    g = torch.Generator(device=dev).manual_seed(B + L + d)
    G = torch.zeros(B, (L + 7) // 8 * 8, device=dev, dtype=torch.float16)
    G[:, :L] = (torch.rand(B, L, generator=g, device=dev) - 0.4).half()
    return G, _normal(dev, B, B, d, d, 0.05, torch.float16)


@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_gradient(dev, beta):
    B, L, d, ld = 128, 60001, 776, 780
    assert L * d > 40 << 20
    G, X = _inputs(dev, B, L, d)
    grad = _normal(dev, 3, L, ld, d, 0.1, torch.float32)
    before = grad.clone()
    if beta == 0.0:
        grad[:, :d] = float("nan")  # what is there is not read
    print(f"gradient: B={B} L={L} d={d} beta={beta}", flush=True)
    check(lib().xfc_dw(G.data_ptr(), G.stride(0), X.data_ptr(), d, grad.data_ptr(), ld, B, L, d, beta, _st()), "xfc_dw")
    for l0 in range(0, L, CHUNK):
        l1 = min(L, l0 + CHUNK)
        dW, aW = _gradient(G, X, d, l0, l1)
        was = beta * before[l0:l1, :d].double()
        assert bool(((grad[l0:l1, :d].double() - dW - was).abs() <= SUM * aW + 2.0 ** -22 * was.abs() + 1e-30).all())
    assert torch.equal(grad[:, d:], before[:, d:])


@pytest.mark.parametrize("state,B,L,least", [("fp16", 8, 200003, 140 << 20), ("fp32", 64, 40003, 28 << 20)])
def test_update(dev, state, B, L, least):
    d = 776
    ld = d + 8
    assert L * d > least
    dtype = torch.float16 if state == "fp16" else torch.float32
    G, X = _inputs(dev, B, L, d)
    W, M = _normal(dev, 1, L, ld, d, 0.02, dtype), _normal(dev, 2, L, ld, d, 0.01, dtype)
    W0, M0 = W.clone(), M.clone()
    print(f"update: {state} B={B} L={L} d={d}", flush=True)
    if state == "fp16":
        check(lib().xfc_dw_update(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), ld, M.data_ptr(), ld, B, L, d, LR, MU, WD, None, 0,
                                  _st()), "xfc_dw_update")
    else:
        half = _normal(dev, 4, L, ld, d, 0.02, torch.float16)
        check(lib().xfc_dw_update_master(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), ld, M.data_ptr(), ld, half.data_ptr(), ld, B, L, d,
                                         LR, MU, WD, None, 0, _st()), "xfc_dw_update_master")
        assert torch.equal(half[:, :d], W[:, :d].half()) and bool((half[:, d:] == 7.0).all())  # the fp16 copy, to the last bit
    rounding = 2.0 ** -11 if state == "fp16" else 2.0 ** -23
    least_step = 2.0 ** -25 if state == "fp16" else 0.0  # half the smallest step of fp16
    for l0 in range(0, L, CHUNK):
        l1 = min(L, l0 + CHUNK)
        dW, aW = _gradient(G, X, d, l0, l1)
        w0, m0 = W0[l0:l1, :d].double(), M0[l0:l1, :d].double()
        m = MU * m0 + dW + WD * w0
        w = w0 - LR * m
        slack = SUM * aW + 2.0 ** -22 * (m0.abs() + w0.abs())
        assert bool(((M[l0:l1, :d].double() - m).abs() <= slack + rounding * m.abs() + least_step).all())
        assert bool(((W[l0:l1, :d].double() - w).abs() <= slack + rounding * w.abs() + least_step).all())
    assert torch.equal(W[:, d:], W0[:, d:]) and torch.equal(M[:, d:], M0[:, d:])
