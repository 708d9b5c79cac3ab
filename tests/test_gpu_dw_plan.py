"""dW by large tiles in each mode and each way of storing, and by small ones past the caches, which the sizes are asserted to lead to: labels
and dims that end inside a tile, rows that end inside a stage.  Checks and bounds are those of test_gpu_dw_tiles.py."""
import pytest
import test_gpu_dw_tiles as tiles
import torch
from test_tile_plan import CACHED, MASTER, OUT, PAST, THROUGH, UPDATE, plans  # noqa: F401

pytestmark = pytest.mark.gpu
LARGE, SMALL = False, True


def _goes_by(plans, size, tile, how):
    assert plans.dw([size], torch.cuda.get_device_properties(0).multi_processor_count) == [(tile, how)]


@pytest.mark.parametrize("B,L,d,tile,how", [(1, 65531, 248, LARGE, THROUGH), (300, 32763, 504, LARGE, THROUGH), (40, 65531, 504, LARGE, CACHED),
                                            (300, 65531, 504, LARGE, CACHED), (63, 65531, 1016, LARGE, PAST), (700, 65533, 760, LARGE, PAST),
                                            (130, 60001, 776, SMALL, PAST)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_gradient(dev, plans, B, L, d, tile, how, beta):  # noqa: F811
    _goes_by(plans, (B, L, d, OUT), tile, how)
    tiles.test_gradient(dev, B, L, d, beta)


@pytest.mark.parametrize("state,B,L,d,tile,how", [
    ("fp16", 65, 65531, 248, LARGE, THROUGH), ("fp16", 63, 65531, 1016, LARGE, CACHED), ("fp16", 8, 163835, 1016, LARGE, PAST),
    ("fp16", 130, 200003, 776, SMALL, PAST), ("fp32", 520, 65531, 184, LARGE, THROUGH), ("fp32", 520, 65531, 248, LARGE, CACHED),
    ("fp32", 520, 65531, 504, LARGE, PAST), ("fp32", 700, 65533, 760, LARGE, PAST), ("fp32", 63, 65531, 504, SMALL, PAST)])
def test_update(dev, plans, state, B, L, d, tile, how):  # noqa: F811
    _goes_by(plans, (B, L, d, UPDATE if state == "fp16" else MASTER), tile, how)
    tiles.test_update(dev, state, B, L, d)
