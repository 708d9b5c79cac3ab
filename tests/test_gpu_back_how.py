"""The joint pass of up to 256 rows by each way of storing what it writes, which the sizes are asserted to lead to, with rows that are whole lines of
128 bytes and rows that are not.  Checks and bounds are those of test_gpu_back_step.py."""
import pytest
import test_gpu_back_step as back
from test_tile_plan import ADD, CACHED, OUT, PAST, THROUGH, UPDATE, plans  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,d,pad,how", [(37, 21001, 768, 64, THROUGH), (200, 10003, 320, 0, THROUGH), (100, 33001, 768, 0, CACHED), (130, 70001, 320, 64, CACHED),
                                           (64, 90001, 448, 64, PAST), (100, 80001, 768, 64, PAST), (150, 300003, 128, 0, PAST), (255, 200001, 192, 64, PAST),
                                           (64, 90001, 448, 8, CACHED), (255, 100001, 392, 0, CACHED), (30, 21001, 776, 56, CACHED), (30, 2001, 776, 0, THROUGH)])
def test_update(dev, plans, B, L, d, pad, how):  # noqa: F811
    assert plans.back([(B, L, d, UPDATE)], d % 64 == 0 and (d + pad) % 64 == 0) == [how]
    back.test_update_in_one_pass(dev, B, L, d, pad)


@pytest.mark.parametrize("B,L,d,pad,how", [(100, 30001, 768, 32, CACHED), (70, 55001, 768, 64, PAST), (200, 130001, 352, 0, PAST), (9, 450003, 96, 32, PAST),
                                           (40, 55001, 776, 0, CACHED), (200, 330001, 352, 4, CACHED)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_accumulation(dev, plans, B, L, d, pad, how, beta):  # noqa: F811
    assert plans.back([(B, L, d, ADD if beta else OUT)], d % 32 == 0 and (d + pad) % 32 == 0) == [how] and not plans.gradients_apart([(B, L, d, beta != 0.0)])[0]
    back.test_accumulation_in_one_pass(dev, B, L, d, pad, beta)


def test_a_gradient_of_pieces_of_lines_past_the_caches(dev, plans):  # noqa: F811
    B, L, d = 130, 60001, 776
    assert plans.back([(B, L, d, OUT)], False) == [PAST]
    back.test_accumulation_in_one_pass(dev, B, L, d, 0, 0.0)
