"""dX and dW (or the update) in one pass, for batches of up to 256 rows, against float64: rows at the edges of its four row
counts, label counts at the edges of a tile of 64 and of G's pieces of eight, widths that do not fill a slice of 128 dims or a
group of 64, leading dimensions past the width, accumulation, and the workspaces it is given.  Bounds: fp32 sums of up to 256
(dW) or L (dX) products of halves, relative to the sums of their magnitudes, 2^-23 per addition with a factor of four for
the order; W and M one rounding to fp16 on top (2^-11)."""
import pytest
import torch

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu
SUM = 4 * 2.0 ** -23


def _st():
    return torch.cuda.current_stream().cuda_stream


def _operands(dev, B, L, d, pad):
    g = torch.Generator().manual_seed(B * 7 + L * 3 + d)
    ldg, ld = (L + 7) // 8 * 8 + 8, d + pad
    G = torch.full((B, ldg), float("nan"))
    G[:, : (L + 7) // 8 * 8] = 0.0            # pad columns up to the next eight are zero, past them never read
    G[:, :L] = torch.rand(B, L, generator=g) - 0.4
    X = torch.full((B, ld), 7.0)
    X[:, :d] = torch.randn(B, d, generator=g) * 0.05
    W = torch.full((L, ld), 9.0)
    W[:, :d] = torch.randn(L, d, generator=g) * 0.02
    M = torch.full((L, ld), 5.0)
    M[:, :d] = torch.randn(L, d, generator=g) * 0.01
    return [t.half().to(dev) for t in (G, X, W, M)]


def _reference(G, X, W, d, L, scale):
    g, x, w = G[:, :L].double(), X[:, :d].double(), W[:, :d].double()
    return scale * (g @ w), scale * (g.abs() @ w.abs()), g.t() @ x, g.abs().t() @ x.abs()


@pytest.mark.parametrize("B,L,d,pad", [(1, 1, 8, 0), (3, 64, 72, 8), (64, 65, 128, 0), (65, 63, 136, 8), (100, 1003, 64, 0),
                                       (128, 4097, 768, 0), (129, 513, 200, 16), (192, 777, 384, 0), (193, 70001, 64, 0),
                                       (199, 9001, 1024, 0), (256, 20011, 768, 8), (255, 130, 120, 0),
                                       (100, 80001, 768, 0),   # too large for the caches: loads and stores with the hint
                                       (48, 1100003, 56, 8),   # loads alone
                                       (49, 950003, 64, 0)])
def test_update_in_one_pass(dev, B, L, d, pad):
    G, X, W, M = _operands(dev, B, L, d, pad)
    lr, mu, wd, scale = 0.1, 0.9, 0.01, 2.0
    dX, aX, dW, aW = _reference(G, X, W, d, L, scale)
    W0, M0 = W[:, :d].double(), M[:, :d].double()
    m = mu * M0 + dW + wd * W0
    w = W0 - lr * m
    full = max(lib().xfc_step_workspace_bytes(B, L, d, 0), 1 << 20)
    for nbytes in (full, 8 * B * d * 4):
        Wt, Mt = W.clone(), M.clone()
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        out = torch.full((B, d + 4), float("nan"), device=dev)
        print(f"update: B={B} L={L} d={d} workspace={nbytes}", flush=True)
        check(lib().xfc_dx_dw_update(G.data_ptr(), G.stride(0), X.data_ptr(), X.stride(0), Wt.data_ptr(), Wt.stride(0),
                                     Mt.data_ptr(), Mt.stride(0), out.data_ptr(), d + 4, B, L, d, lr, mu, wd, scale,
                                     ws.data_ptr(), nbytes, _st()), "xfc_dx_dw_update")
        assert bool(((out[:, :d].double() - dX).abs() <= SUM * aX + 1e-30).all())
        assert bool(torch.isnan(out[:, d:]).all())
        slack = SUM * aW + 2.0 ** -22 * (M0.abs() + W0.abs())
        assert bool(((Mt[:, :d].double() - m).abs() <= slack + 2.0 ** -11 * m.abs() + 2.0 ** -25).all())
        assert bool(((Wt[:, :d].double() - w).abs() <= slack + 2.0 ** -11 * w.abs() + 2.0 ** -25).all())
        assert torch.equal(Wt[:, d:], W[:, d:]) and torch.equal(Mt[:, d:], M[:, d:])


@pytest.mark.parametrize("B,L,d,pad", [(2, 5, 8, 0), (64, 129, 72, 8), (128, 1003, 768, 0), (190, 64, 136, 0), (256, 5001, 384, 4),
                                       (257, 1003, 64, 0), (70, 55001, 768, 0)])
@pytest.mark.parametrize("beta", [0.0, 1.0, 0.5])
def test_accumulation_in_one_pass(dev, B, L, d, pad, beta):
    G, X, W, _ = _operands(dev, B, L, d, 0)
    scale = 0.5
    dX, aX, dW, aW = _reference(G, X, W, d, L, scale)
    grad0 = torch.randn(L, d + pad, generator=torch.Generator().manual_seed(1)).to(dev)
    if beta == 0.0:
        grad0[:] = float("nan")   # not read
    grad = grad0.clone()
    want = dW + (beta * grad0[:, :d].double() if beta else 0.0)
    nbytes = lib().xfc_step_workspace_bytes(B, L, d, 0)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    out = torch.empty(B, d, device=dev)
    Wt = W.clone()
    print(f"accumulate: B={B} L={L} d={d} beta={beta}", flush=True)
    check(lib().xfc_dx_dw(G.data_ptr(), G.stride(0), X.data_ptr(), X.stride(0), Wt.data_ptr(), Wt.stride(0), grad.data_ptr(),
                          d + pad, out.data_ptr(), d, B, L, d, beta, scale, ws.data_ptr(), nbytes, _st()), "xfc_dx_dw")
    assert bool(((out.double() - dX).abs() <= SUM * aX + 1e-30).all())
    assert bool(((grad[:, :d].double() - want).abs() <= SUM * aW + 2.0 ** -22 * want.abs() + 1e-30).all())
    assert torch.equal(Wt, W) and torch.equal(grad[:, d:].nan_to_num(), grad0[:, d:].nan_to_num())


def test_what_the_two_calls_refuse_is_refused(dev):
    G, X, W, M = _operands(dev, 70, 200, 64, 0)
    dX = torch.empty(70, 64, device=dev)
    ws = torch.empty(8 * 70 * 64 * 4, dtype=torch.uint8, device=dev)

    def call(ldg=None, nbytes=ws.numel(), m=None):
        return lib().xfc_dx_dw_update(G.data_ptr(), G.stride(0) if ldg is None else ldg, X.data_ptr(), 64, W.data_ptr(), 64,
                                      M.data_ptr() if m is None else None, 64, dX.data_ptr(), 64, 70, 200, 64, 0.1, 0.9, 0.0, 1.0,
                                      ws.data_ptr(), nbytes, _st())
    assert call(ldg=196) == 3                     # not a multiple of 8
    assert call(ldg=192) == 6                     # shorter than the labels
    assert call(nbytes=ws.numel() - 16) == 4      # less than 8 partial sums
    assert call(m=0) == 1                         # no momentum
    assert call() == 0


# the last: more partial sums than ranges, which only wide or very long operands have
@pytest.mark.parametrize("B,L,d", [(128, 131072, 768), (199, 131072, 768), (256, 320001, 384), (256, 40001, 1024), (5, 60007, 3072)])
def test_dx_is_as_close_to_float64_as_by_itself(dev, B, L, d):
    """The sums of dX may not be longer than xfc_dx's: their error (of random roundings, so with some allowance for chance, a
    tenth) against float64 is the measure.  G all of one sign, as after the first steps, W not."""
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
    check(lib().xfc_dx_dw_update(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), d, M.data_ptr(), d, one.data_ptr(), d, B, L, d,
                                 0.0, 0.9, 0.0, 1.0, ws.data_ptr(), ws.numel(), _st()), "xfc_dx_dw_update")
    error = [float((t.double() - want).norm() / want.norm()) for t in (one, two)]
    print(f"  {error[0]:.2e}, xfc_dx {error[1]:.2e}", flush=True)
    assert not torch.equal(one, two)  # the joint pass has run, and not the two in its place
    assert error[0] <= 1.1 * error[1]


@pytest.mark.parametrize("B,L,d", [(192, 560007, 768), (100, 131072, 384), (48, 60007, 512)])
def test_gradients_that_take_two_passes(dev, B, L, d):
    """129 to 256 rows of 768 dims on a long axis and 33 to 128 of middle sizes: the two passes, which are faster there, to the
    last bit."""
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    G = torch.zeros(B, (L + 7) // 8 * 8, dtype=torch.float16, device=dev)
    G[:, :L] = torch.rand(B, L, generator=g, device=dev)
    X = torch.randn(B, d, generator=g, device=dev).half()
    W = torch.randn(L, d, generator=g, device=dev).half()
    ws = torch.empty(max(lib().xfc_step_workspace_bytes(B, L, d, 0), lib().xfc_dx_workspace_bytes(B, L, d)), dtype=torch.uint8, device=dev)
    dX, grad = torch.empty(2, B, d, device=dev), torch.empty(2, L, d, device=dev)
    check(lib().xfc_dx_dw(G.data_ptr(), G.stride(0), X.data_ptr(), d, W.data_ptr(), d, grad[0].data_ptr(), d, dX[0].data_ptr(), d, B, L, d,
                          0.0, 1.0, ws.data_ptr(), ws.numel(), _st()), "xfc_dx_dw")
    check(lib().xfc_dx(G.data_ptr(), G.stride(0), W.data_ptr(), d, dX[1].data_ptr(), d, B, L, d, 1.0, ws.data_ptr(), ws.numel(), _st()), "xfc_dx")
    check(lib().xfc_dw(G.data_ptr(), G.stride(0), X.data_ptr(), d, grad[1].data_ptr(), d, B, L, d, 0.0, _st()), "xfc_dw")
    assert torch.equal(dX[0], dX[1]) and torch.equal(grad[0], grad[1])
