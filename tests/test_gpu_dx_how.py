"""dX by itself by both ways of storing its partial sums, with rows of these that are whole lines and that are not, against float64.  Checks and
bounds are those of test_gpu_through.py."""
import pytest
import test_gpu_through as through
from test_tile_plan import CACHED, THROUGH, plans  # noqa: F401

from renee_amd._lib import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,d,how", [(200, 1001, 200, CACHED), (129, 9001, 136, CACHED), (600, 4001, 776, CACHED), (257, 3001, 160, THROUGH),
                                       (512, 1001, 128, THROUGH), (300, 1001, 72, THROUGH), (128, 9001, 776, THROUGH), (300, 4001, 768, THROUGH)])
def test_gradient_of_the_input(dev, plans, B, L, d, how):  # noqa: F811
    assert plans.dx([(B, L, d, lib().xfc_dx_workspace_bytes(B, L, d))], d % 32 == 0) == [how]
    through.test_gradient_of_the_input(dev, B, L, d)
