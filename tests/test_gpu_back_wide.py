"""dX and the update in one pass for 257 to 512 rows, against float64: rows at the edges of its four row counts and of the eights it
fetches, label counts at the edges of a tile of 64, of its halves and of G's pieces of eight, fewer tiles than ranges and more, with and
without the hint for sizes that no cache holds, from the first labels on and from the last, leading dimensions past the width, and the
calls that it leaves to the two passes.  Bounds: fp32 sums of up to 512 (dW) or L (dX) products of halves, relative to the sums of their magnitudes, 2^-23 per addition with
a factor of four for the order; W and M one rounding to fp16 on top (2^-11)."""
import pytest
import torch
from test_gpu_back_step import SUM, _operands, _reference, _st

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _call(G, X, W, M, out, ws, B, L, d, lr=0.1, mu=0.9, wd=0.01, scale=2.0):
    return lib().xfc_dx_dw_update(G.data_ptr(), G.stride(0), X.data_ptr(), X.stride(0), W.data_ptr(), W.stride(0), M.data_ptr(), M.stride(0),
                                  out.data_ptr(), out.stride(0), B, L, d, lr, mu, wd, scale, ws.data_ptr(), ws.numel(), _st())


@pytest.mark.parametrize("B,L,d,pad", [(257, 1, 128, 0), (264, 31, 128, 8), (320, 32, 256, 0), (321, 33, 128, 8), (383, 63, 128, 0),
                                       (384, 64, 384, 0), (385, 65, 128, 8), (448, 95, 256, 0), (449, 97, 128, 0), (505, 1003, 768, 8),
                                       (511, 2753, 768, 0), (512, 4096, 1024, 0), (512, 129, 3072, 0), (300, 20011, 128, 0),
                                       (512, 40009, 256, 8),
                                       (290, 65001, 768, 0),    # more than the caches hold: non-temporal loads, the last
                                       (512, 80001, 768, 8)])   # labels first
def test_update_in_one_pass(dev, B, L, d, pad):
    _update(dev, B, L, d, pad)


@pytest.mark.parametrize("whole", [1, 31, 33, 48])
@pytest.mark.parametrize("B,d", [(320, 256), (384, 256), (400, 256), (512, 256), (449, 384)])
def test_the_tile_that_is_not_whole_comes_first(dev, B, d, whole):
    """Where the pass runs from the last labels on, with more than the Infinity Cache holds: the first tile has 1 to 48 labels and
    another one follows it."""
    L = (150_000 if d < 384 else 120_000) // 64 * 64 + whole
    assert 224 << 20 < L * (4 * d + 2 * B)
    _update(dev, B, L, d, 0)


def _update(dev, B, L, d, pad):
    G, X, W, M = _operands(dev, B, L, d, pad)
    lr, mu, wd, scale = 0.1, 0.9, 0.01, 2.0
    dX, aX, dW, aW = _reference(G, X, W, d, L, scale)
    W0, M0 = W[:, :d].double(), M[:, :d].double()
    m = mu * M0 + dW + wd * W0
    w = W0 - lr * m
    Wt, Mt = W.clone(), M.clone()
    ws = torch.empty(lib().xfc_step_workspace_bytes(B, L, d, 0), dtype=torch.uint8, device=dev)
    out = torch.full((B, d + 4), float("nan"), device=dev)
    print(f"update: B={B} L={L} d={d}", flush=True)
    check(_call(G, X, Wt, Mt, out, ws, B, L, d, lr, mu, wd, scale), "xfc_dx_dw_update")
    assert bool(((out[:, :d].double() - dX).abs() <= SUM * aX + 1e-30).all())
    assert bool(torch.isnan(out[:, d:]).all())
    slack = SUM * aW + 2.0 ** -22 * (M0.abs() + W0.abs())
    assert bool(((Mt[:, :d].double() - m).abs() <= slack + 2.0 ** -11 * m.abs() + 2.0 ** -25).all())
    assert bool(((Wt[:, :d].double() - w).abs() <= slack + 2.0 ** -11 * w.abs() + 2.0 ** -25).all())
    assert torch.equal(Wt[:, d:], W[:, d:]) and torch.equal(Mt[:, d:], M[:, d:])


def test_values_that_are_not_finite_stay_in_their_rows_labels_and_dims(dev):
    """A row of G, a label of W and M and a column of X, in a batch whose last rows share an image with rows that are none."""
    B, L, d = 300, 1003, 256
    G, X, W, M = _operands(dev, B, L, d, 0)
    G[299, 5], G[17, 1002], W[64, 3], M[77, 9], X[260, 200] = float("inf"), float("nan"), float("-inf"), float("nan"), float("inf")
    ws = torch.empty(lib().xfc_step_workspace_bytes(B, L, d, 0), dtype=torch.uint8, device=dev)
    out = torch.empty(B, d, device=dev)
    Wt, Mt = W.clone(), M.clone()
    check(_call(G, X, Wt, Mt, out, ws, B, L, d), "xfc_dx_dw_update")
    dx_ok, m_ok = torch.ones(B, d, dtype=torch.bool, device=dev), torch.ones(L, d, dtype=torch.bool, device=dev)
    dx_ok[299], dx_ok[17], dx_ok[:, 3] = False, False, False
    m_ok[5], m_ok[1002], m_ok[64, 3], m_ok[77, 9], m_ok[:, 200] = False, False, False, False, False
    assert torch.equal(torch.isfinite(out), dx_ok)
    assert torch.equal(torch.isfinite(Mt), m_ok) and torch.equal(torch.isfinite(Wt), m_ok)


@pytest.mark.parametrize("B,L,d", [(512, 131072, 768), (300, 20011, 256), (400, 320001, 384), (257, 131072, 3072)])  # the last: parts
def test_dx_is_as_close_to_float64_as_by_itself(dev, B, L, d):
    """As for fewer rows: the sums of dX may not be longer than xfc_dx's, a tenth for chance."""
    g = torch.Generator(device=dev)
    g.manual_seed(B + L)
    G = torch.zeros(B, (L + 7) // 8 * 8, dtype=torch.float16, device=dev)
    G[:, :L] = torch.rand(B, L, generator=g, device=dev)
    X = torch.randn(B, d, generator=g, device=dev).half()
    W = (torch.randn(L, d, generator=g, device=dev) * 0.02).half()
    M = torch.zeros_like(W)
    want = torch.zeros(B, d, dtype=torch.float64, device=dev)
    for l0 in range(0, L, 16384):
        want += G[:, l0:min(L, l0 + 16384)].double() @ W[l0:l0 + 16384].double()
    ws = torch.empty(max(lib().xfc_step_workspace_bytes(B, L, d, 0), lib().xfc_dx_workspace_bytes(B, L, d)), dtype=torch.uint8, device=dev)
    one, two = torch.empty(B, d, device=dev), torch.empty(B, d, device=dev)
    print(f"dX: B={B} L={L} d={d}", flush=True)
    check(lib().xfc_dx(G.data_ptr(), G.stride(0), W.data_ptr(), d, two.data_ptr(), d, B, L, d, 1.0, ws.data_ptr(), ws.numel(), _st()), "xfc_dx")
    check(_call(G, X, W, M, one, ws, B, L, d, 0.0, 0.9, 0.0, 1.0), "xfc_dx_dw_update")
    error = [float((t.double() - want).norm() / want.norm()) for t in (one, two)]
    print(f"  {error[0]:.2e}, xfc_dx {error[1]:.2e}", flush=True)
    assert not torch.equal(one, two)  # the joint pass has run, and not the two in its place
    assert error[0] <= 1.1 * error[1]


@pytest.mark.parametrize("why", ["width", "strides", "workspace", "rows"])
def test_calls_that_take_two_passes(dev, why):
    """Widths that are no multiple of 128, a momentum with another leading dimension, a short workspace, more rows: to the last bit."""
    B, L, d = 513 if why == "rows" else 300, 20011, 192 if why == "width" else 256
    G, X, W, M = _operands(dev, B, L, d, 0)
    if why == "strides":
        M = torch.nn.functional.pad(M, (0, 8))
    full = max(lib().xfc_step_workspace_bytes(B, L, d, 0), lib().xfc_dx_workspace_bytes(B, L, d))
    ws = torch.empty(8 * B * d * 4 if why == "workspace" else full, dtype=torch.uint8, device=dev)
    out, W2, M2 = torch.empty(2, B, d, device=dev), torch.stack([W, W]), torch.stack([M, M])
    check(_call(G, X, W2[0], M2[0], out[0], ws, B, L, d), "xfc_dx_dw_update")
    check(lib().xfc_dx(G.data_ptr(), G.stride(0), W2[1].data_ptr(), d, out[1].data_ptr(), d, B, L, d, 2.0, ws.data_ptr(), ws.numel(), _st()), "xfc_dx")
    check(lib().xfc_dw_update(G.data_ptr(), G.stride(0), X.data_ptr(), d, W2[1].data_ptr(), d, M2[1].data_ptr(), M.stride(0), B, L, d, 0.1, 0.9,
                              0.01, None, 0, _st()), "xfc_dw_update")
    assert torch.equal(out[0], out[1]) and torch.equal(W2[0], W2[1]) and torch.equal(M2[0], M2[1])
