"""dW by large and small tiles in each mode and each way of storing, which the sizes are asserted to lead to: labels and dims that end inside a
tile, rows that end inside a stage, rows that are whole lines of 128 bytes and rows that are not, leading dimensions past the width; against
float64.  Bounds are those of test_gpu_past_caches.py."""
import pytest
import torch
from test_gpu_back_step import SUM, _st
from test_gpu_past_caches import LR, MU, WD, _gradient, _inputs, _normal
from test_tile_plan import CACHED, MASTER, OUT, PAST, THROUGH, UPDATE, plans  # noqa: F401

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu
LARGE, SMALL = False, True
CHUNK = 1 << 15


def _goes_by(plans, mode, B, L, d, pad, tile, how):
    row = 64 if mode == UPDATE else 32  # elements of a line
    whole = d % row == 0 and (d + pad) % row == 0
    assert plans.dw([(B, L, d, mode)], torch.cuda.get_device_properties(0).multi_processor_count, whole) == [(tile, how)]


@pytest.mark.parametrize("B,L,d,pad,tile,how", [
    (1, 65531, 192, 64, LARGE, THROUGH), (300, 32763, 480, 0, LARGE, THROUGH), (40, 65531, 448, 32, LARGE, CACHED), (63, 65531, 960, 0, LARGE, PAST),
    (700, 65533, 704, 64, LARGE, PAST), (130, 60001, 800, 0, SMALL, PAST), (70, 3001, 96, 32, SMALL, THROUGH), (300, 65531, 1016, 8, LARGE, CACHED),
    (130, 60001, 776, 4, SMALL, CACHED), (33, 300001, 200, 0, LARGE, CACHED), (16, 3001, 768, 4, SMALL, THROUGH)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_gradient(dev, plans, B, L, d, pad, tile, how, beta):  # noqa: F811
    _goes_by(plans, OUT, B, L, d, pad, tile, how)
    ld = d + pad
    G, X = _inputs(dev, B, L, d)
    grad = _normal(dev, 3, L, ld, d, 0.1, torch.float32)
    before = grad.clone()
    if beta == 0.0:
        grad[:, :d] = float("nan")  # what is there is not read
    print(f"gradient: B={B} L={L} d={d} ld={ld} beta={beta}", flush=True)
    check(lib().xfc_dw(G.data_ptr(), G.stride(0), X.data_ptr(), d, grad.data_ptr(), ld, B, L, d, beta, _st()), "xfc_dw")
    for l0 in range(0, L, CHUNK):
        l1 = min(L, l0 + CHUNK)
        dW, aW = _gradient(G, X, d, l0, l1)
        was = beta * before[l0:l1, :d].double()
        assert bool(((grad[l0:l1, :d].double() - dW - was).abs() <= SUM * aW + 2.0 ** -22 * was.abs() + 1e-30).all())
    assert torch.equal(grad[:, d:], before[:, d:])


@pytest.mark.parametrize("mode,B,L,d,pad,tile,how", [
    (UPDATE, 65, 65531, 192, 64, LARGE, THROUGH), (UPDATE, 63, 65531, 960, 0, LARGE, CACHED), (UPDATE, 8, 163835, 960, 64, LARGE, PAST),
    (UPDATE, 130, 200003, 832, 0, SMALL, PAST), (UPDATE, 33, 4001, 128, 64, SMALL, THROUGH), (UPDATE, 63, 65531, 1016, 8, LARGE, CACHED),
    (UPDATE, 16, 300001, 136, 0, LARGE, CACHED), (UPDATE, 600, 200003, 776, 8, SMALL, CACHED), (UPDATE, 70, 3001, 776, 0, SMALL, THROUGH),
    (MASTER, 520, 65531, 192, 0, LARGE, THROUGH), (MASTER, 520, 65531, 256, 32, LARGE, CACHED), (MASTER, 520, 65531, 480, 32, LARGE, PAST),
    (MASTER, 700, 65533, 704, 0, LARGE, PAST), (MASTER, 63, 70003, 448, 64, SMALL, PAST), (MASTER, 35, 451991, 256, 0, LARGE, PAST),
    (MASTER, 520, 65531, 504, 8, LARGE, CACHED), (MASTER, 16, 196003, 200, 8, LARGE, CACHED), (MASTER, 40, 30001, 776, 0, SMALL, CACHED)])
def test_update(dev, plans, mode, B, L, d, pad, tile, how):  # noqa: F811
    _goes_by(plans, mode, B, L, d, pad, tile, how)
    ld = d + pad
    dtype = torch.float16 if mode == UPDATE else torch.float32
    G, X = _inputs(dev, B, L, d)
    W, M = _normal(dev, 1, L, ld, d, 0.02, dtype), _normal(dev, 2, L, ld, d, 0.01, dtype)
    W0, M0 = W.clone(), M.clone()
    print(f"update: {dtype} B={B} L={L} d={d} ld={ld}", flush=True)
    if mode == UPDATE:
        check(lib().xfc_dw_update(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), ld, M.data_ptr(), ld, B, L, d, LR, MU, WD, None, 0,
                                  _st()), "xfc_dw_update")
    else:
        half = _normal(dev, 4, L, ld, d, 0.02, torch.float16)
        check(lib().xfc_dw_update_master(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), ld, M.data_ptr(), ld, half.data_ptr(), ld, B, L, d,
                                         LR, MU, WD, None, 0, _st()), "xfc_dw_update_master")
        assert torch.equal(half[:, :d], W[:, :d].half()) and bool((half[:, d:] == 7.0).all())  # the fp16 copy, to the last bit
    rounding = 2.0 ** -11 if mode == UPDATE else 2.0 ** -23
    least_step = 2.0 ** -25 if mode == UPDATE else 0.0  # half the smallest step of fp16
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
