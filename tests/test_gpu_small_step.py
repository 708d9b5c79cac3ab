"""The one-pass step of batches up to 64 rows against the three passes that larger batches take, which a workspace
without room for its partial sums selects: same labels, same G.  z is summed in another order, so results are compared
within what rounding G, the weights and the momentum to fp16 allows (2^-11 of each value, once) and never bit by bit."""
import pytest
import torch

from renee_amd import XFCLayer, synth
from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _step(dev, X, W, M, rp, ci, coo, scale, ldg, ws_bytes):
    h, (B, d), L = lib(), X.shape, W.shape[0]
    W, M = W.to(dev).clone(), M.to(dev).clone()
    G = torch.full((B + 1, ldg), 7.0, dtype=torch.float16, device=dev)
    dX = torch.full((B, d + 4), 3.0, device=dev)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    if coo:
        px = torch.repeat_interleave(torch.arange(B), (rp[1:] - rp[:-1]).long()).to(dev)
        py, name, nnz = ci.long().to(dev), "xfc_step_coo", ci.numel()
        pairs = (px, py)
    else:
        pairs, name, nnz = (rp.to(dev), ci.to(dev)), "xfc_step_csr", ci.numel()
    rc = getattr(h, name)(X.data_ptr(), X.stride(0), W.data_ptr(), d, M.data_ptr(), d, pairs[0].data_ptr(),
                          pairs[1].data_ptr(), nnz, G.data_ptr(), ldg, dX.data_ptr(), d + 4, B, L, d, 0.05, 0.9, 1e-4,
                          scale, ws.data_ptr(), ws.numel(), st)
    check(rc, name)
    torch.cuda.synchronize()
    return G, dX, W, M


# one row, both row tiles and their edges; each width; one label, a partial tile, a count that is no multiple of 8, several
# tiles to a workgroup
@pytest.mark.parametrize("B,L,d", [(1, 1, 128), (16, 33, 256), (32, 4097, 768), (33, 1000, 768), (64, 40001, 768),
                                   (31, 70003, 128), (64, 70001, 128), (64, 20000, 256), (17, 30011, 384),
                                   (49, 30011, 384), (32, 9001, 512), (64, 20007, 512), (32, 20001, 1024), (5, 31, 1024)])
@pytest.mark.parametrize("coo", [False, True])
def test_one_pass_matches_three(dev, B, L, d, coo):
    h = lib()
    check(h.xfc_init(), "xfc_init")
    X = synth.make_X(B, d, 7).half().to(dev)
    W = (synth.make_W(L, d, 7) * 3).half()
    M = torch.empty(L, d).normal_(0.0, 1e-2, generator=torch.Generator().manual_seed(L)).half()
    P = synth.make_positives(B, L, min(8, L), 1.0 + min(2.0, L - 1), 1.1, 7)
    rp, ci = torch.from_numpy(P.rowptr).int(), torch.from_numpy(P.colidx).int()
    ldg = (L + 7) // 8 * 8 + 8
    full = h.xfc_step_workspace_bytes(B, L, d, ci.numel())
    fwd = (h.xfc_fwd_grad_workspace_bytes(L, ci.numel()) + 255) // 256 * 256
    small = fwd + 8 * B * d * 4   # the three passes on the fewest slices of the label axis
    tiles = ((L + 7) // 8 * 8 + 31) // 32
    print(f"one pass: B={B} L={L} d={d} coo={coo}", flush=True)
    G, dX, Wn, Mn = _step(dev, X, W, M, rp, ci, coo, 2.0, ldg, full)
    if tiles > 8:  # below that both workspaces hold the one pass
        G3, dX3, W3, M3 = _step(dev, X, W, M, rp, ci, coo, 2.0, ldg, small)
        assert not torch.equal(dX, dX3) or B == 1   # two different routes
        assert torch.equal(G[:B, :L] < 0, G3[:B, :L] < 0)
    Xd, Wd, Md = X.double().cpu(), W.double(), M.double()
    Z = Xd @ Wd.t()
    Y = torch.zeros(B, L, dtype=torch.float64)
    Y[torch.repeat_interleave(torch.arange(B), (rp[1:] - rp[:-1]).long()), ci.long()] = 1.0
    want_G = torch.sigmoid(Z) - Y
    assert (G[:B, :L].double().cpu() - want_G).abs().max() <= 2.0 ** -11 + 1e-5   # |G| <= 1
    assert bool((G[:B, L:(L + 7) // 8 * 8] == 0).all()) and bool((G[:B, (L + 7) // 8 * 8:] == 7).all())
    assert bool((G[B:] == 7).all())
    Gd = G[:B, :L].double().cpu()    # the products are those of the rounded G: fp32 sums
    want = 2.0 * Gd @ Wd
    assert (dX[:, :d].double().cpu() - want).norm() <= 1e-5 * want.norm()
    assert bool((dX[:, d:] == 3.0).all())
    m = 0.9 * Md + (Gd.t() @ Xd + 1e-4 * Wd)
    w = Wd - 0.05 * m
    assert ((Mn.double().cpu() - m).abs() <= 2.0 ** -11 * m.abs() + 1e-5).all()
    assert ((Wn.double().cpu() - w).abs() <= 2.0 ** -11 * w.abs() + 1e-5).all()


# a thread holds 4, 8, 4 and 3 pairs (three times 768 threads overhang the 2048)
@pytest.mark.parametrize("B,d", [(32, 256), (32, 128), (50, 512), (50, 384)])
def test_one_pass_label_lists(dev, B, d):
    """Pairs out of range are dropped, one listed twice counts once, and lists longer than the workgroups hold (2048) or
    empty give the same step."""
    L = 5000
    X, W = synth.make_X(B, d, 8).half().to(dev), synth.make_W(L, d, 8).half()
    g = torch.Generator().manual_seed(1)
    for n, extra in ((0, 0), (3, 3), (2048, 0), (2049, 0)):
        px, py = torch.randint(0, B, (n,), generator=g), torch.randint(0, L, (n,), generator=g)
        if extra:
            px = torch.cat([px, px, torch.tensor([-1, B, 0, 1])])
            py = torch.cat([py, py, torch.tensor([3, 3, -1, L])])
        lay = XFCLayer(L, d, B, dev, weight=W, max_positives=4096)
        print(f"label list of {px.numel()}", flush=True)
        lay.xfc_backward(X, px.to(dev), py.to(dev))
        Y = torch.zeros(B, L, dtype=torch.bool)
        keep = (px >= 0) & (px < B) & (py >= 0) & (py < L)
        Y[px[keep], py[keep]] = True
        assert torch.equal((lay.outsoft[:B, :L] < 0).cpu(), Y)
        want = torch.sigmoid(X.double().cpu() @ W.double().t()) - Y.double()
        assert (lay.outsoft[:B, :L].double().cpu() - want).abs().max() <= 2.0 ** -11 + 1e-5


# rows past the batch in the first or the second 16 of a pair, both row tiles
@pytest.mark.parametrize("B,d", [(20, 128), (50, 768), (9, 1024)])
def test_one_pass_infinite_weight_stays_in_its_label_and_dim(dev, B, d):
    L = 300
    X, W = synth.make_X(B, d, 9).half().to(dev), synth.make_W(L, d, 9).half()
    W[70, 5] = float("inf")
    lay = XFCLayer(L, d, B, dev, weight=W)
    dX = lay.xfc_backward(X, torch.zeros(1, dtype=torch.int64, device=dev), torch.zeros(1, dtype=torch.int64, device=dev))
    cols = torch.arange(d) != 5
    assert bool(torch.isfinite(dX[:, cols]).all()) and not bool(torch.isfinite(dX[:, 5]).all())
    rows = torch.arange(L) != 70
    assert bool(torch.isfinite(lay.xfc_weight[rows]).all()) and bool(torch.isfinite(lay.outsoft[:B, :L]).all())
    # the other dims of that label are updated as those of any other, in fp32 and rounded once
    Gd = lay.outsoft[:B, :L].double().cpu()
    m = Gd.t() @ X.double().cpu()
    w = W.double() - 0.05 * m
    for got, want in ((lay.momentum_buffer, m), (lay.xfc_weight, w)):
        got = got.double().cpu()
        assert bool(torch.isfinite(got[70, cols]).all())
        assert ((got - want).abs() <= 2.0 ** -11 * want.abs() + 1e-5)[:, cols].all()
