"""dW by tiles of 128 labels x 128 dims and of 256 x 256, whichever the sizes lead to: the update, its form with master weights, and the
gradient, written and added to, at labels, dims and rows at the edges of both tiles and of a stage of 64 rows, leading dimensions past
the width, against float64.  Bounds are those of test_gpu_past_caches.py."""
import pytest
import torch
from test_gpu_back_step import SUM, _st
from test_gpu_past_caches import LR, MU, WD, _gradient, _inputs, _normal

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu
SIZES = [(1, 1, 8), (63, 127, 120), (64, 129, 128), (65, 128, 136), (130, 257, 200), (300, 1000, 264), (700, 385, 1024), (1030, 20003, 768),
         (1024, 33001, 256)]


@pytest.mark.parametrize("B,L,d", SIZES)
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_gradient(dev, B, L, d, beta):
    ld = d + 4
    G, X = _inputs(dev, B, L, d)
    grad = _normal(dev, 3, L, ld, d, 0.1, torch.float32)
    before = grad.clone()
    if beta == 0.0:
        grad[:, :d] = float("nan")  # what is there is not read
    print(f"gradient: B={B} L={L} d={d} beta={beta}", flush=True)
    check(lib().xfc_dw(G.data_ptr(), G.stride(0), X.data_ptr(), d, grad.data_ptr(), ld, B, L, d, beta, _st()), "xfc_dw")
    dW, aW = _gradient(G, X, d, 0, L)
    was = beta * before[:, :d].double()
    assert bool(((grad[:, :d].double() - dW - was).abs() <= SUM * aW + 2.0 ** -22 * was.abs() + 1e-30).all())
    assert torch.equal(grad[:, d:], before[:, d:])


@pytest.mark.parametrize("B,L,d", SIZES)
@pytest.mark.parametrize("state", ["fp16", "fp32"])
def test_update(dev, state, B, L, d):
    ld = d + 8
    dtype = torch.float16 if state == "fp16" else torch.float32
    G, X = _inputs(dev, B, L, d)
    W, M = _normal(dev, 1, L, ld, d, 0.02, dtype), _normal(dev, 2, L, ld, d, 0.01, dtype)
    W0, M0 = W.clone(), M.clone()
    dump = _normal(dev, 5, L, d + 4, d, 0.0, torch.float32)
    print(f"update: {state} B={B} L={L} d={d}", flush=True)
    if state == "fp16":
        check(lib().xfc_dw_update(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), ld, M.data_ptr(), ld, B, L, d, LR, MU, WD,
                                  dump.data_ptr(), d + 4, _st()), "xfc_dw_update")
    else:
        half = _normal(dev, 4, L, ld, d, 0.02, torch.float16)
        check(lib().xfc_dw_update_master(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), ld, M.data_ptr(), ld, half.data_ptr(), ld, B, L, d,
                                         LR, MU, WD, dump.data_ptr(), d + 4, _st()), "xfc_dw_update_master")
        assert torch.equal(half[:, :d], W[:, :d].half()) and bool((half[:, d:] == 7.0).all())  # the fp16 copy, to the last bit
    dW, aW = _gradient(G, X, d, 0, L)
    assert bool(((dump[:, :d].double() - dW).abs() <= SUM * aW + 1e-30).all()) and bool((dump[:, d:] == 7.0).all())
    rounding = 2.0 ** -11 if state == "fp16" else 2.0 ** -23
    least_step = 2.0 ** -25 if state == "fp16" else 0.0  # half the smallest step of fp16
    w0, m0 = W0[:, :d].double(), M0[:, :d].double()
    m = MU * m0 + dW + WD * w0
    w = w0 - LR * m
    slack = SUM * aW + 2.0 ** -22 * (m0.abs() + w0.abs())
    assert bool(((M[:, :d].double() - m).abs() <= slack + rounding * m.abs() + least_step).all())
    assert bool(((W[:, :d].double() - w).abs() <= slack + rounding * w.abs() + least_step).all())
    assert torch.equal(W[:, d:], W0[:, d:]) and torch.equal(M[:, d:], M0[:, d:])
