"""dX and a gradient that is written or added to on both sides of the lines between the joint pass and two passes, which the sizes are asserted to
lie on, against float64.  Checks and bounds are those of test_gpu_back_step.py."""
import pytest
import test_gpu_back_step as back
import torch
from test_tile_plan import plans  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,d,adds,apart", [(16, 95003, 512, 0, False), (33, 50003, 1024, 1, False), (64, 62805, 768, 0, False),
                                              (9, 180005, 256, 1, False), (9, 850003, 64, 0, True), (48, 150003, 64, 1, True),
                                              (64, 230003, 256, 0, True)])
def test_both_gradients(dev, plans, B, L, d, adds, apart):  # noqa: F811
    assert plans.gradients_apart([(B, L, d, adds)], torch.cuda.get_device_properties(0).multi_processor_count) == [apart]
    for beta in ((0.5, 1.0) if adds else (0.0,)):
        back.test_accumulation_in_one_pass(dev, B, L, d, 0, beta)


# longest chains of sums: the joint pass at sizes that took two until now
@pytest.mark.parametrize("B,L,d", [(5, 1000003, 768), (33, 700001, 1024), (64, 320001, 512)])
def test_dx_is_as_close_to_float64_as_by_itself(dev, B, L, d):
    back.test_dx_is_as_close_to_float64_as_by_itself(dev, B, L, d)
