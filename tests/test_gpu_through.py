"""Updates, gradients and partial sums of dX on both sides of the sizes up to which they are written through the L2, against float64, with leading
dimensions past the width.  Checks and bounds are those of test_gpu_back_step.py and test_gpu_past_caches.py."""
import pytest
import test_gpu_back_step as back
import test_gpu_dw_tiles as tiles
import test_gpu_past_caches as past
import torch
from test_gpu_back_step import _st

from renee_amd._lib import check, lib

pytestmark = pytest.mark.gpu
Mi = 1 << 20


@pytest.mark.parametrize("B,L,d", [(37, 21001, 768), (200, 22001, 768)])  # 64 MiB of weights and momentum lie between
def test_joint_update(dev, B, L, d):
    back.test_update_in_one_pass(dev, B, L, d, 8)


@pytest.mark.parametrize("state,B,L,least", [("fp16", 16, 60001, 44 * Mi), ("fp16", 16, 66001, 48 * Mi), ("fp32", 16, 16001, 11 * Mi),
                                             ("fp32", 16, 17001, 12 * Mi), ("fp32", 16, 701, 0)])
def test_update(dev, state, B, L, least):
    past.test_update(dev, state, B, L, least)


# 16 and 40 Mi weights lie between, the latter on large tiles up to 48 rows
@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("B,L,d", [(16, 21001, 768), (16, 22001, 768), (700, 22001, 768), (48, 320001, 128), (48, 340001, 128), (56, 340001, 128)])
def test_gradient(dev, B, L, d, beta):
    tiles.test_gradient(dev, B, L, d, beta)


@pytest.mark.parametrize("B,L,d", [(40, 3001, 64), (130, 8001, 72), (600, 1001, 200), (512, 33001, 768), (140, 200001, 256),
                                   (130, 39999, 72), (130, 40001, 72)])  # 48 MiB of partial sums, 40,000 labels
def test_gradient_of_the_input(dev, B, L, d):
    g = torch.Generator(device=dev).manual_seed(B + L)
    G = torch.zeros(B, (L + 7) // 8 * 8, dtype=torch.float16, device=dev)
    G[:, :L] = (torch.rand(B, L, generator=g, device=dev) - 0.4).half()
    W = (torch.randn(L, d, generator=g, device=dev) * 0.02).half()
    ws = torch.full((lib().xfc_dx_workspace_bytes(B, L, d),), 255, dtype=torch.uint8, device=dev)
    dX = torch.full((B, d + 4), 7.0, device=dev)
    print(f"dX: B={B} L={L} d={d} partial sums {ws.numel() >> 20} MiB", flush=True)
    check(lib().xfc_dx(G.data_ptr(), G.stride(0), W.data_ptr(), d, dX.data_ptr(), d + 4, B, L, d, 0.5, ws.data_ptr(), ws.numel(), _st()), "xfc_dx")
    want, mag = torch.zeros(B, d, dtype=torch.float64, device=dev), torch.zeros(B, d, dtype=torch.float64, device=dev)
    for l0 in range(0, L, 1 << 14):
        x, w = G[:, l0:min(L, l0 + (1 << 14))].double(), W[l0:l0 + (1 << 14)].double()
        want += x @ w
        mag += x.abs() @ w.abs()
    assert bool(((dX[:, :d].double() - 0.5 * want).abs() <= 0.5 * back.SUM * mag + 1e-30).all()) and bool((dX[:, d:] == 7.0).all())
