"""The forward pass by each of its plans, which the sizes are asserted to lead to: tiles of 64 and 128 rows, large and small tiles of the
wide loop, and large ones with the labels after whole rounds of them by small ones; rows, labels and dims at their edges, few logits and
many, the loss with a workspace that is aligned and one that is not.  Checks and bounds are those of test_gpu_fwd_tiles.py."""
import pytest
import test_gpu_fwd_tiles as tiles
import torch
from test_tile_plan import plans  # noqa: F401

from renee_amd import xfc_gemm
from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu
# rows, labels, dims, which tile, whether small ones follow (without the loss and with it)
SIZES = [(1, 257, 200, "64", (0, 0)), (40, 4001, 72, "64", (0, 0)), (64, 30001, 64, "64", (0, 0)),
         (65, 65529, 64, "128", (0, 0)), (100, 40001, 72, "128", (0, 0)), (128, 65535, 200, "128", (0, 0)),
         (512, 131001, 64, "wide", (0, 0)), (256, 65535, 72, "wide", (0, 0)),
         (256, 32761, 64, "wide128", (0, 0)), (1024, 8185, 72, "wide128", (0, 0)), (300, 131071, 64, "wide128", (0, 0)),
         (512, 131073, 768, "wide", (1, 1)), (385, 80003, 1024, "wide", (1, 1)), (255, 150001, 1024, "wide", (1, 1)),
         (1000, 40005, 1024, "wide", (1, 1))]


def _cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def _goes_by(plans, size, tile, rest):
    got = plans.forward([size], _cus())[0]
    assert got[0] == tile and (got[4] > 0) == bool(rest), got


@pytest.mark.parametrize("B,L,d,tile,rest", SIZES)
def test_logits_gradient_and_loss(dev, plans, B, L, d, tile, rest):  # noqa: F811
    n_store = (L + 7) // 8 * 8
    for loss in (0, 1):
        _goes_by(plans, (B, n_store, d, loss), tile, rest[loss])
    _goes_by(plans, (B, L, d, 0), tile, rest[0])
    tiles.test_logits_gradient_and_loss(dev, B, L, d)

    # the loss again in a workspace that is not aligned, which has places for fewer partial sums
    X, W, z, az = tiles._inputs(dev, B, L, d)
    nbytes = lib().xfc_fwd_grad_workspace_bytes(L, 0)
    ws = torch.full((nbytes + 4,), 255, dtype=torch.uint8, device=dev)
    G, loss = torch.empty(B, n_store, device=dev, dtype=torch.float16), torch.full((1,), float("nan"), device=dev)
    check(lib().xfc_fwd_grad_coo(X.data_ptr(), d + 8, W.data_ptr(), d + 8, None, None, 0, G.data_ptr(), n_store, B, L, d, loss.data_ptr(),
                                 ws.data_ptr() + 4, nbytes, tiles._st()), "xfc_fwd_grad_coo")
    want = float(torch.nn.functional.softplus(z).sum())
    assert abs(float(loss) - want) <= float((tiles.SUM * az + 2.0 ** -21).sum()) + 2.0 ** -23 * want
    assert tiles._rounded(G[:, :L], torch.sigmoid(z), 0.25 * tiles.SUM * az + 2.0 ** -21)


@pytest.mark.parametrize("B,L,d,tile,rest", [(40, 4008, 72, "64", 0), (100, 40008, 72, "128", 0), (128, 60008, 64, "128", 0),
                                             (512, 131000, 64, "wide", 0), (385, 80008, 1024, "wide", 1)])
def test_alpha_and_beta(dev, plans, B, L, d, tile, rest):  # noqa: F811
    _goes_by(plans, (B, L, d, 0), tile, rest)
    X, W, z, az = tiles._inputs(dev, B, L, d, 0)
    for beta in (0.0, 0.5):
        out = torch.rand(B, L, device=dev).half()
        want = torch.sigmoid(0.5 * z + beta * out.double())
        print(f"sigmoid: B={B} L={L} d={d} beta={beta}", flush=True)
        xfc_gemm(X, W.t(), out, 0.5, beta, True)
        assert tiles._rounded(out, want, 0.25 * (0.5 * tiles.SUM * az + 2.0 ** -22) + 2.0 ** -21)


# with the maxima of blocks of 32
@pytest.mark.parametrize("B,L,d,tile,rest", [(64, 90001, 64, "64", 0), (128, 65537 - 8, 72, "128", 0), (512, 131073, 768, "wide", 1),
                                             (385, 80003, 1024, "wide", 1), (255, 150001, 1024, "wide", 1)])
def test_best_of_the_logits(dev, plans, B, L, d, tile, rest):  # noqa: F811
    _goes_by(plans, (B, L, d, 0), tile, rest)
    tiles.test_best_of_the_logits(dev, B, L, d)
