"""The loss from the forward pass (dl_base.py:578-583) where its parts are much larger than itself: a learnt positive, whose
term softplus(z) - z is the small rest of two large numbers, and a sum of many equal terms.  Against float64, on all three
row tiles."""
import math

import pytest
import torch

from renee_amd import XFCLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [40, 100, 300])
def test_term_of_a_learnt_positive(dev, B):
    """One positive at z = 10, everything else at z = -30, whose terms are below 1e-12 each.  The term is 4.5e-5; what it
    may be off by is the rounding of 1 + e^-z, 2^-24, and those of the logarithm and the result, well below that again."""
    L, d = 777, 768
    g = torch.Generator().manual_seed(B)
    code = torch.where(torch.rand(B, d, generator=g) < 0.5, -1.0, 1.0) / math.sqrt(d - 1)
    code[:, 0] = 1.0
    X = code.half()
    for row, label in ((0, 0), (1, 776), (B - 1, 255), (B // 2, 256), (17, 511), (31, 700), (32, 33), (B - 2, 3)):
        W = torch.zeros(L, d)
        W[:, 0] = -30.0
        W[label, 1:] = 40.0 * (1.0 + row / B / 100) * code[row, 1:]   # not the same z for every row
        W = W.half()
        lay = XFCLayer(L, d, B, dev, weight=W)
        loss = torch.zeros(1, device=dev)
        pair = (torch.tensor([row], device=dev), torch.tensor([label], device=dev))
        print(f"learnt positive: B={B} row={row} label={label}", flush=True)
        lay.fwd_grad(X.to(dev), *pair, loss_out=loss)
        Z = X.double() @ W.double().t()
        Y = torch.zeros(B, L, dtype=torch.float64)
        Y[row, label] = 1.0
        want = float(torch.nn.functional.softplus(torch.where(Y > 0, -Z, Z)).sum())
        assert 1e-5 < want < 1e-4
        assert abs(float(loss) - want) <= 2.0 ** -23


# every row tile, many tiles to a workgroup
@pytest.mark.parametrize("B,L", [(64, 600_000), (128, 600_000), (512, 600_001)])
def test_sum_of_many_equal_terms(dev, B, L):
    """All logits zero: B . L . log 2, which sums in fp32 over a workgroup's tiles miss by 1e-6 and more.  Each group of
    terms and the result are rounded to fp32 once (2^-24), and log 2 itself."""
    d = 8
    lay = XFCLayer(L, d, B, dev, weight=torch.zeros(L, d).half())
    loss = torch.zeros(1, device=dev)
    print(f"equal terms: B={B} L={L}", flush=True)
    lay.fwd_grad(torch.ones(B, d, device=dev).half(), None, None, loss_out=loss)
    want = B * L * math.log(2.0)
    assert abs(float(loss) - want) <= 2.0 ** -22 * want
